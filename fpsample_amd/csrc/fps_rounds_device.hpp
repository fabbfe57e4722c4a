// fps_rounds_device.hpp -- device parts shared by the threshold-round kernels.
#pragma once
#include "fps_device.hpp"
#include "fps_rounds.hpp"
#include "fps_rounds_bound.hpp"

namespace fpsx {

template <int TIE>
__device__ __forceinline__ uint32_t tie_of(uint32_t idx) {
  return TIE == kTieHighest ? idx : ~idx;
}

// Wave-wide maximum of a 64-bit key (uniform).
__device__ __forceinline__ uint64_t wave_max_u64(uint64_t k) {
  const uint32_t hi = wave_max_u32((uint32_t)(k >> 32));
  const uint32_t lo = wave_max_u32((uint32_t)(k >> 32) == hi ? (uint32_t)k : 0u);
  return ((uint64_t)hi << 32) | lo;
}

__device__ __forceinline__ uint32_t lanes_below(uint64_t mask) {
  return __builtin_amdgcn_mbcnt_hi((uint32_t)(mask >> 32),
                                   __builtin_amdgcn_mbcnt_lo((uint32_t)mask, 0u));
}

__device__ __forceinline__ uint64_t readlane_u64(uint64_t v, int lane) {
  return ((uint64_t)(uint32_t)readlane_i((int)(v >> 32), lane) << 32) |
         (uint32_t)readlane_i((int)(uint32_t)v, lane);
}

__device__ __forceinline__ uint32_t uniform_u32(uint32_t v) {
  return (uint32_t)__builtin_amdgcn_readfirstlane((int)v);
}

__device__ __forceinline__ uint64_t uniform_u64(uint64_t v) {
  return ((uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)(v >> 32)) << 32) |
         (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)v);
}

// A launch's parameters where the scalar unit reads them.  A round reads what it needs again
// (a kernel argument kept over the whole loop holds scalar registers, which then spill).
typedef const __attribute__((address_space(4))) RoundsParams *ParamsPtr;

// One record of a candidate's coordinates in LDS, read 16 bytes at a time.
template <int D>
struct alignas(16) Rec {
  float c[D > 0 ? (D + 3) / 4 * 4 : 4];
};

// Reports a failure (one thread).
__device__ __forceinline__ void rounds_fail(ParamsPtr a, uint32_t code) {
  atomicOr(a->fps.status, code);
  if (a->host_status)
    __hip_atomic_store(a->host_status, code, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

// Counters of a workgroup's rounds in LDS.
struct RoundsCounts {
  uint32_t cnt[2];  // candidates of this workgroup, by round parity
  uint32_t sum[2];  // candidates of the grid, by round parity
  uint32_t at[2];   // candidates taken in, by round parity
  uint64_t wmax[kRoundsThreads / 64];  // best key of every wave
  uint64_t te[2];   // keys that the round's picks must exceed beside its bound, by round parity
  uint32_t stop[2]; // first pick that does not lower itself, by round parity
  uint32_t np[2];   // picks, by round parity
  uint64_t step;    // the next round's step
  uint64_t last;    // key of the last pick where the run is cut there
  uint32_t stuck;
  uint32_t ok;

  __device__ __forceinline__ void clear(int parity) {
    cnt[parity] = sum[parity] = at[parity] = 0;
    te[parity] = 0;
    stop[parity] = ~0u;
    np[parity] = 0;
  }
};

// The exchange of round e: own candidates (keys lk, coordinates lc) out, everybody's into ck and
// cc in any order.  On return C is the number of all (more than LIST where they do not fit) and,
// where it is that or 0, U the best key of all.  False when something did not arrive in time.  Entered
// and left by all waves, with a barrier before it is left.
// L lanes read one workgroup's header and its first L candidates at once, so most candidates
// are here as soon as their header is; those beyond L follow, a memory round trip later (64
// workgroups at L = 2, 4, 8 and 16: 50 K points 807, 711, 665 and 664 us a run, 100 K x 6-D
// 1247, 1029, 938 and 914; 16 workgroups at 8, 16 and 32, 4096 points: 256, 243 and 240).  NC
// coordinates go with a key.
template <int NC, int LIST>
__device__ __forceinline__ bool rounds_exchange(uint64_t *xchg, uint64_t spin_ticks, uint32_t capw,
                                                uint32_t G, uint32_t g, uint32_t e, int tid,
                                                int wave, RoundsCounts &S, const uint64_t *lk,
                                                const Rec<NC> *lc, uint64_t *ck, Rec<NC> *cc,
                                                uint32_t &C, uint64_t &U) {
  constexpr uint32_t NWC = 2 + NC;
  constexpr int W = kRoundsThreads / 64;
  const int lane = tid & 63;
  const uint32_t par = e & 1u;
  const uint32_t own = C;
  const uint32_t hp = rounds_head_pitch(G);
  const size_t head = (size_t)kRoundsReplicas * kRoundsHeadWords * hp;
  const size_t cp = (size_t)G * capw;  // pitch of one word's array
  uint64_t *buf = xchg + (size_t)par * (head + NWC * cp);
  uint64_t *cbuf = buf + head;
  if (wave == 0) {
    if (lane < (int)(kRoundsReplicas * kRoundsHeadWords)) {
      const uint32_t rep = (uint32_t)lane / kRoundsHeadWords;
      const uint32_t k = (uint32_t)lane - rep * kRoundsHeadWords;
      const uint32_t v = k == 0 ? own : (k == 1 ? (uint32_t)(U >> 32) : (uint32_t)U);
      xchg_store(buf + ((size_t)rep * kRoundsHeadWords + k) * hp + g,
                 ((uint64_t)v << 32) | e);
    }
  } else if (own <= capw) {
    for (uint32_t q = (uint32_t)tid - 64; q < own; q += kRoundsThreads - 64) {
      const uint64_t k = lk[q];
      uint64_t *w = cbuf + (size_t)g * capw + q;
      xchg_store(w, (k & 0xffffffff00000000ull) | e);
      xchg_store(w + cp, (k << 32) | e);
      if constexpr (NC > 0) {
        const Rec<NC> r = lc[q];
#pragma unroll
        for (int j = 0; j < NC; ++j)
          xchg_store(w + (size_t)(2 + j) * cp,
                     ((uint64_t)(uint32_t)__float_as_int(r.c[j]) << 32) | e);
      }
    }
  }
  const uint32_t shift = G <= 32 ? 5 : G <= 64 ? 4 : G <= 128 ? 3 : 2;
  const uint32_t L = 1u << shift;
  const uint32_t q = (uint32_t)tid >> shift;
  const uint32_t l = (uint32_t)tid & (L - 1);
  if ((uint32_t)wave * 64 < G * L) {
    const uint64_t *h =
        buf + (size_t)(g % kRoundsReplicas) * kRoundsHeadWords * hp + q;
    const uint64_t *w = cbuf + (size_t)q * capw;
    uint32_t cq = 0;
    uint64_t v[NWC];
    const bool mine = q < G;
    bool here = false;  // candidate l of workgroup q is there
    if (mine) {
      const uint64_t deadline = now_ticks() + spin_ticks;
      for (;;) {
        const uint64_t w0 = xchg_load(h);
#pragma unroll
        for (uint32_t k = 0; k < NWC; ++k) v[k] = xchg_load(w + l + k * cp);
        bool all = true;
#pragma unroll
        for (uint32_t k = 0; k < NWC; ++k) all = all && (uint32_t)v[k] == e;
        cq = (uint32_t)(w0 >> 32);
        here = l < cq && cq <= capw;
        if ((uint32_t)w0 == e && (all || !here)) break;
        if (now_ticks() > deadline) {
          S.ok = 0;
          cq = 0;
          here = false;
          break;
        }
      }
    }
    const uint32_t sum =
        (uint32_t)__builtin_amdgcn_readlane((int)wave_scan_add(l == 0 ? cq : 0u), 63);
    if (lane == 0 && sum) atomicAdd(&S.sum[par], sum);
    uint32_t i = l;
    for (;;) {
      const uint64_t m = __ballot(here);
      if (!m) break;
      uint32_t at = 0;
      if (lane == 0) at = atomicAdd(&S.at[par], (uint32_t)__popcll(m));
      at = (uint32_t)__builtin_amdgcn_readfirstlane((int)at) + lanes_below(m);
      if (here && at < (uint32_t)LIST) {
        ck[at] = (v[0] & 0xffffffff00000000ull) | (v[1] >> 32);
        if constexpr (NC > 0) {
          Rec<NC> r;
#pragma unroll
          for (int j = 0; j < NC; ++j) r.c[j] = __int_as_float((int)(v[2 + j] >> 32));
          cc[at] = r;
        }
      }
      i += L;
      here = here && i < cq;
      if (here) {
        const uint64_t deadline = now_ticks() + spin_ticks;
        for (;;) {
          bool all = true;
#pragma unroll
          for (uint32_t k = 0; k < NWC; ++k) v[k] = xchg_load(w + i + k * cp);
#pragma unroll
          for (uint32_t k = 0; k < NWC; ++k) all = all && (uint32_t)v[k] == e;
          if (all) break;
          if (now_ticks() > deadline) {
            S.ok = 0;
            here = false;
            break;
          }
        }
      }
    }
  }
  lds_barrier();
  if (!__builtin_amdgcn_readfirstlane((int)S.ok)) return false;
  C = S.sum[par];
  const uint32_t got = S.at[par];
  if (got != C || C > (uint32_t)LIST) C = max(C, (uint32_t)LIST + 1);  // some did not fit
  if (C == 0 || C > (uint32_t)LIST) {
    // No candidates to decide on: the best key of all, read only now, is the pick.
    uint64_t u = 0;
    for (uint32_t i = (uint32_t)tid; i < G; i += kRoundsThreads) {
      const uint64_t *h = buf + ((size_t)(g % kRoundsReplicas) * kRoundsHeadWords + 1) * hp + i;
      const uint64_t deadline = now_ticks() + spin_ticks;
      for (;;) {
        const uint64_t w1 = xchg_load(h), w2 = xchg_load(h + hp);
        if ((uint32_t)w1 == e && (uint32_t)w2 == e) {
          u = (w1 & 0xffffffff00000000ull) | (w2 >> 32);
          break;
        }
        if (now_ticks() > deadline) {
          S.ok = 0;
          break;
        }
      }
    }
    u = wave_max_u64(u);
    if (lane == 0) S.wmax[wave] = u;
    lds_barrier();
    if (!uniform_u32(S.ok)) return false;
    U = wave_max_u64(lane < W ? S.wmax[lane] : 0ull);
  }
  return true;
}

// Adds to rank[i] how many of the C keys exceed key i (ck is 0 beyond C, up to the next
// multiple of 16; rank starts at 0).  A job is 32 keys against 16, eight for each half of the
// wave, so that a last piece of few keys costs little.  The comparison is a subtraction's
// borrow, added with carry: three instructions a pair and no 64-bit compare (the compiler
// makes that compare again of __builtin_subc).
__device__ __forceinline__ void rank_candidates(const uint64_t *ck, uint32_t *rank, uint32_t C,
                                                int tid, int wave) {
  const int lane = tid & 63;
  constexpr int W = kRoundsThreads / 64;
  const uint32_t nc = (C + 31u) >> 5;
  const uint32_t nj = (C + 15u) >> 4;
  uint32_t ic = wave;
  uint32_t jc = 0;
  while (ic >= nc) {
    ic -= nc;
    ++jc;
  }
  while (jc < nj) {
    const uint32_t i = ic * 32 + (lane & 31);
    const uint64_t ki = ck[i];
    const uint64_t *kj = ck + jc * 16 + (lane >> 5) * 8;
    uint32_t r = 0;
#pragma unroll
    for (int l = 0; l < 8; ++l) {
      const uint64_t k = kj[l];
      uint32_t t;
      asm("v_sub_co_u32 %1, vcc, %2, %3\n\t"
          "v_subb_co_u32 %1, vcc, %4, %5, vcc\n\t"
          "v_addc_co_u32 %0, vcc, 0, %0, vcc"
          : "+v"(r), "=&v"(t)
          : "v"((uint32_t)ki), "v"((uint32_t)k), "v"((uint32_t)(ki >> 32)), "v"((uint32_t)(k >> 32))
          : "vcc");
    }
    if (i < C && r) atomicAdd(&rank[i], r);
    ic += W;
    while (ic >= nc) {
      ic -= nc;
      ++jc;
    }
  }
}

// The picks among F sorted candidates, were no candidate only partly lowered: each one that no
// earlier pick lowers, settled in a few steps per 64 candidates rather than one by one.  rows:
// bits of the earlier candidates that lower candidate i, 32 a word at [word][CAP].  One wave.
template <int CAP>
__device__ __forceinline__ void settle_candidates(const uint32_t *rows, uint32_t F, int lane,
                                                  uint64_t *out) {
  constexpr int CH = CAP / 64;
  const uint32_t nc = (F + 63u) >> 6;
  uint64_t low[CH][CH];
#pragma unroll
  for (int c = 0; c < CH; ++c)
#pragma unroll
    for (int w = 0; w <= c; ++w)
      low[c][w] = ((uint64_t)rows[(2 * w + 1) * CAP + c * 64 + lane] << 32) |
                  rows[2 * w * CAP + c * 64 + lane];
  uint64_t acc[CH];
#pragma unroll
  for (int c = 0; c < CH; ++c) {
    acc[c] = 0;
    if ((uint32_t)c < nc) {
      uint64_t before = 0;
#pragma unroll
      for (int w = 0; w < c; ++w) before |= low[c][w] & acc[w];
      const uint64_t same = low[c][c] & (((uint64_t)1 << lane) - 1);
      uint64_t open = __ballot((uint32_t)(c * 64 + lane) < F && before == 0);
      while (open) {
        const uint64_t free = __ballot((same & open) == 0) & open;
        acc[c] |= free;
        open &= ~free;
        open &= ~__ballot((same & free) != 0);
      }
    }
    if (lane == 0) out[c] = acc[c];
  }
}

}  // namespace fpsx
