// fps_rounds.hip -- exact farthest point sampling in threshold rounds.
//
// The vanilla loop (reference src/lib.cpp:188-246) takes one pick per pass over the
// cloud.  Min-distances only ever fall, so a whole run of picks can be taken from few
// points: let every point have the key (min-distance, index) whose maximum is the next
// pick, and let T be any bound.  The points whose key exceeds T are the candidates.  While
// the best candidate's current key exceeds T, it is the best point of the whole cloud (every
// other point's key was at most T and has not risen), so the picks come from the candidates
// alone.  One round is then
//   1. update: every block of 64 * P points takes the last round's picks, skipping those too
//      far from the block's bounding box to change its largest min-distance, and hands in
//      its points above the new T;
//   2. exchange: every workgroup publishes its candidates and reads everybody's;
//   3. front: every workgroup derives the same picks from the same candidates: they are
//      sorted by key and taken in order.  A pick that lowers a later candidate takes that
//      candidate out of the order; should its new key still exceed T, T rises to it, so
//      the round ends before that candidate would have to be placed anew.
// T is the last bound minus a step in key space; the step follows the number of candidates.
// Keys are total (the index breaks ties), so steps below one value work through any number
// of equal distances.
//
// What bounds it: a round's serial chain, not bytes (2^20 clustered points, 16384 picks, 128
// workgroups: 224 rounds of 9.5 us).  Of a round (100 K points, 64 workgroups, 363 rounds of
// 9.5 us): update 2.2 us with the wait for the slowest wave, exchange 2.9, sorting 1.4, rows
// 1.9 (the vector ALUs are busy throughout: 10 instructions for 64 pairs), settling 0.4, the
// bound and the picks 1.1.  Settling the candidates one by one instead took 450 ns a pick.
// A block per wave in registers, the candidates loaded beside the headers and the best 256
// taken from up to 512 brought gauss1m from 2.67 to 2.13 ms, 100 K / 50 K picks from 4.52 to
// 3.44 ms.
#include "fps_rounds.hpp"

#include "fps_device.hpp"
#include "fps_kernels.hpp"

namespace fpsx {

namespace {

__device__ __forceinline__ uint64_t make_key(int value_bits, uint32_t tie) {
  return ((uint64_t)((uint32_t)value_bits + 1u) << 32) | tie;
}
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

__device__ __forceinline__ uint64_t uniform_u64(uint64_t v) {
  return ((uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)(v >> 32)) << 32) |
         (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)v);
}

}  // namespace

// One record of a candidate's coordinates in LDS, read 16 bytes at a time.
template <int D>
struct alignas(16) Rec {
  float c[(D + 3) / 4 * 4];
};

// LDS of a workgroup beside its blocks' boxes and best keys.
template <int D>
struct RoundsLds {
  static constexpr int CAP = (int)kRoundsCap;    // candidates the front decides on
  static constexpr int LIST = (int)kRoundsList;  // candidates that may come in
  static constexpr int W = kRoundsThreads / 64;
  alignas(16) uint64_t ck[LIST];  // candidates as they came
  Rec<D> cc[LIST];
  Rec<D> pk[CAP];                 // picks of the round
  uint32_t pt[CAP];               // their tie words
  uint32_t rank[LIST];
  uint64_t sk[CAP];               // sorted candidates
  Rec<D> sc[CAP];
  uint16_t low[CAP / 32][CAP][2];  // rows: which earlier candidates lower this one
  uint64_t lk[CAP];                // this workgroup's candidates
  Rec<D> lc[CAP];
  uint32_t cnt[2];  // candidates of this workgroup, by round parity
  uint32_t sum[2];  // candidates of the grid, by round parity
  uint32_t at[2];   // candidates taken in, by round parity
  uint64_t wmax[W];
  uint64_t acc[CAP / 64];
  uint64_t te;    // the bound that the round's picks exceed
  uint32_t stop;  // first pick that does not lower itself
  uint64_t last;  // key of the round's last pick
  uint32_t np;
  uint32_t stuck;
  uint32_t ok;
};

// Workgroup `group` of G working on one cloud: picks a.s_begin .. a.s_end - 1.
template <int D, int P, int TIE>
__device__ __forceinline__ void rounds_cloud(const RoundsParams &a, const uint32_t group,
                                             const uint32_t G, RoundsLds<D> &S, uint64_t *s_dyn) {
  constexpr int W = RoundsLds<D>::W;
  constexpr int CAP = RoundsLds<D>::CAP;
  constexpr int LIST = RoundsLds<D>::LIST;
  constexpr int CH = CAP / 64;
  constexpr uint32_t NWC = 2 + D;
  const FpsParams &f = a.fps;
  int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const uint32_t nbl = (a.nblocks - group + G - 1) / G;  // blocks group, group + G, ...
  const bool resident = nbl <= (uint32_t)W;          // a block per wave stays in registers
  uint64_t *s_bkey = s_dyn;
  float *s_box = (float *)(s_dyn + nbl);  // [2 * D][nbl]

  if (tid == 0) {
    S.last = ~0ull;
    S.cnt[0] = S.cnt[1] = 0;
    S.sum[0] = S.sum[1] = 0;
    S.at[0] = S.at[1] = 0;
    S.stuck = 0;
    S.ok = 1;
  }

  if (a.s_begin) lds_barrier();  // (a fresh run has one after its forced picks)

  uint32_t s = a.s_begin;  // picks recorded
  uint32_t np = 0;         // picks of the last round, in S.pk
  bool first = true;       // the blocks have not been read yet
  bool last = false;       // the picks are made: apply them and save
  uint64_t T = ~0ull;    // every point's key is at most T
  uint64_t Tg = ~0ull;   // the round's bound
  uint64_t step = (uint64_t)1 << 51;  // a sixteenth of a binade
  if (a.s_begin) {
    // A run taken up again: no key exceeds that of its last pick.
    T = uniform_u64(((uint64_t)a.carry[0] << 32) | a.carry[1]);
    step = uniform_u64(((uint64_t)a.carry[2] << 32) | a.carry[3]);
    Tg = T > step ? T - step : 0;
  }
  uint32_t e = 0;        // rounds
  uint32_t idle = 0;     // rounds since the last pick
  float x[P][D], dm[P];  // the block in hand
  uint32_t id[P];

  for (;;) {
    // Rewritten each round: addresses formed from them would otherwise be kept in registers
    // over the whole loop, beside the block.
    asm volatile("" : "+v"(tid));
    uint32_t g = (uint32_t)__builtin_amdgcn_readfirstlane((int)group);
    asm volatile("" : "+s"(g));
    const int lane = tid & 63;
    // ---- forced picks, in pieces of CAP -------------------------------------
    if (s < f.n_starts) {
      np = min(f.n_starts - s, (uint32_t)CAP);
      if ((uint32_t)tid < np) {
        uint64_t idx = f.starts ? f.starts[s + tid] : a.start;
        if (idx >= f.n) {
          atomicOr(f.status, kStatusBadStart);
          idx = 0;
        }
#pragma unroll
        for (int j = 0; j < D; ++j) S.pk[tid].c[j] = f.pts[(size_t)idx * f.sp + (size_t)j * f.ld];
        S.pt[tid] = tie_of<TIE>((uint32_t)idx);
      }
      lds_barrier();
    }
    // ---- record -------------------------------------------------------------
    if (g == 0) {
      if ((uint32_t)tid < np) {
        f.out[s + tid] = tie_of<TIE>(S.pt[tid]);
        if (f.out_pts != nullptr) {
#pragma unroll
          for (int j = 0; j < D; ++j) f.out_pts[(size_t)(s + tid) * D + j] = S.pk[tid].c[j];
        }
      }
      if (tid == 0) f.status[1] = e;
    }
    s += np;
    if (s >= f.m) return;
    if (s >= a.s_end) {
      last = true;
      if (g == 0 && tid == 0) {
        a.carry[0] = (uint32_t)(S.last >> 32);
        a.carry[1] = (uint32_t)S.last;
        a.carry[2] = (uint32_t)(step >> 32);
        a.carry[3] = (uint32_t)step;
      }
    } else if (np && __builtin_amdgcn_readfirstlane((int)S.stuck)) {
      // The last pick left its own key unchanged, so it stays the best for good.
      if (g == 0) {
        const uint32_t t = S.pt[np - 1];
        for (uint32_t q = s + tid; q < a.s_end; q += kRoundsThreads) {
          f.out[q] = tie_of<TIE>(t);
          if (f.out_pts != nullptr) {
#pragma unroll
            for (int j = 0; j < D; ++j) f.out_pts[(size_t)q * D + j] = S.pk[np - 1].c[j];
          }
        }
      }
      if (a.s_end >= f.m) return;
      last = true;  // (the picks so far are applied below; repeating the last changes nothing)
      if (g == 0 && tid == 0) {
        a.carry[0] = a.carry[1] = ~0u;
        a.carry[2] = (uint32_t)(step >> 32);
        a.carry[3] = (uint32_t)step;
      }
    }
    const bool gather = s >= f.n_starts && !last;  // no further forced picks
    if (!gather) Tg = ~0ull;

    // ---- 1. update ----------------------------------------------------------
    const int tv = (int)(uint32_t)(Tg >> 32) - 1;  // value bits of the bound (-1: below all)
    const uint32_t tt = (uint32_t)Tg;
    const uint32_t nch = (np + 63u) >> 6;
    uint64_t wmax = 0;
    for (uint32_t lb = wave; lb < nbl; lb += W) {
      const uint32_t base = (lb * G + g) * (uint32_t)(64 * P);
      uint64_t hit[CH];
#pragma unroll
      for (int c = 0; c < CH; ++c) hit[c] = 0;
      uint64_t bkey = 0;
      bool any = first || last;
      if (first) {
#pragma unroll
        for (int c = 0; c < CH; ++c) {
          const uint32_t left = np > (uint32_t)(c * 64) ? np - c * 64 : 0u;
          hit[c] = left >= 64 ? ~0ull : (((uint64_t)1 << left) - 1);
        }
      } else {
        bkey = uniform_u64(s_bkey[lb]);
        const float bmax = __int_as_float((int)(uint32_t)(bkey >> 32) - 1);
        float lo[D], hi[D];
#pragma unroll
        for (int j = 0; j < D; ++j) {
          lo[j] = s_box[(uint32_t)j * nbl + lb];
          hi[j] = s_box[(uint32_t)(D + j) * nbl + lb];
        }
#pragma unroll
        for (int c = 0; c < CH; ++c) {
          if ((uint32_t)c < nch) {
            const Rec<D> r = S.pk[c * 64 + lane];
            float p[D];
#pragma unroll
            for (int j = 0; j < D; ++j) p[j] = r.c[j];
            hit[c] = __ballot((uint32_t)(c * 64 + lane) < np && box_bound<D>(p, lo, hi) < bmax);
            any = any || hit[c] != 0;
          }
        }
      }
      if (any || bkey > Tg) {
        if (first || !resident) {
#pragma unroll
          for (int k = 0; k < P; ++k) {
            const uint32_t p = base + (uint32_t)(k * 64 + lane);
            const uint32_t pc = min(p, f.n - 1);
            if (a.rec) {
              const float4 r = a.rec[pc];
              const float r3[3] = {r.x, r.y, r.z};
#pragma unroll
              for (int j = 0; j < D; ++j)
                x[k][j] = j < 3 ? r3[j < 3 ? j : 0] : a.rest[(size_t)(j - 3) * f.n + pc];
              id[k] = (uint32_t)__float_as_int(r.w);
            } else {
#pragma unroll
              for (int j = 0; j < D; ++j) x[k][j] = f.pts[(size_t)pc * f.sp + (size_t)j * f.ld];
              id[k] = pc;
            }
            dm[k] = first && a.s_begin == 0 ? f.init : f.dmin[pc];
          }
          if (base + 64 * P > f.n) {
#pragma unroll
            for (int k = 0; k < P; ++k)
              if (base + (uint32_t)(k * 64 + lane) >= f.n) dm[k] = -1.0f;
          }
        }
        if (first) {
          // Bounding box (clamped padding repeats the last point).
#pragma unroll
          for (int j = 0; j < D; ++j) {
            float lo = INFINITY, hi = -INFINITY;
#pragma unroll
            for (int k = 0; k < P; ++k) {
              lo = fminf(lo, x[k][j]);
              hi = fmaxf(hi, x[k][j]);
            }
            lo = wave_min_f(lo);
            hi = wave_max_f(hi);
            if (lane == 0) {
              s_box[(uint32_t)j * nbl + lb] = lo;
              s_box[(uint32_t)(D + j) * nbl + lb] = hi;
            }
          }
        }
        if (any) {
#pragma unroll
          for (int c = 0; c < CH; ++c) {
            uint64_t mm = hit[c];
            if (mm) {
              const Rec<D> r = S.pk[c * 64 + lane];
              do {
                const int l = __ffsll((unsigned long long)mm) - 1;
                mm &= mm - 1;
                float p[D];
#pragma unroll
                for (int j = 0; j < D; ++j) p[j] = readlane_f(r.c[j], l);
#pragma unroll
                for (int k = 0; k < P; ++k) dm[k] = min_keep(sqdist<D>(x[k], p), dm[k]);
              } while (mm);
            }
          }
          if (!resident || last) {
#pragma unroll
            for (int k = 0; k < P; ++k) {
              const uint32_t p = base + (uint32_t)(k * 64 + lane);
              if (p < f.n) f.dmin[p] = dm[k];
            }
          }
          // The block's best key.
          int bv = INT_MIN;
#pragma unroll
          for (int k = 0; k < P; ++k) bv = max(bv, __float_as_int(dm[k]));
          const int wv = wave_max_i32(bv);
          uint32_t bt = 0;
#pragma unroll
          for (int k = 0; k < P; ++k)
            if (__float_as_int(dm[k]) == wv) bt = max(bt, tie_of<TIE>(id[k]));
          const uint64_t tied = __ballot(bv == wv);
          const uint32_t wt = __popcll(tied) == 1
                                  ? (uint32_t)readlane_i((int)bt, __ffsll((unsigned long long)tied) - 1)
                                  : wave_max_u32(bt);
          bkey = make_key(wv, wt);
          if (lane == 0) s_bkey[lb] = bkey;
        }
        if (bkey > Tg) {
          uint64_t m[P];
          uint32_t total = 0;
#pragma unroll
          for (int k = 0; k < P; ++k) {
            const int b = __float_as_int(dm[k]);
            m[k] = __ballot(b > tv || (b == tv && tie_of<TIE>(id[k]) > tt));
            total += (uint32_t)__popcll(m[k]);
          }
          uint32_t at = 0;
          if (lane == 0) at = atomicAdd(&S.cnt[(e + 1) & 1], total);
          at = (uint32_t)__builtin_amdgcn_readfirstlane((int)at);
#pragma unroll
          for (int k = 0; k < P; ++k) {
            const uint32_t q = at + lanes_below(m[k]);
            if (((m[k] >> lane) & 1) && q < (uint32_t)CAP) {
              S.lk[q] = make_key(__float_as_int(dm[k]), tie_of<TIE>(id[k]));
              Rec<D> r;
#pragma unroll
              for (int j = 0; j < D; ++j) r.c[j] = x[k][j];
              S.lc[q] = r;
            }
            at += (uint32_t)__popcll(m[k]);
          }
        }
      }
      wmax = bkey > wmax ? bkey : wmax;
    }
    first = false;
    if (last) return;
    if (!gather) {
      lds_barrier();
      continue;
    }
    if (lane == 0) S.wmax[wave] = wmax;
    if (tid < LIST) {
      S.ck[tid] = 0;
      S.rank[tid] = 0;
    }
    if (tid == 0) {
      S.te = Tg;
      S.stop = ~0u;
    }
    lds_barrier();
    ++e;
    const uint32_t par = e & 1u;
    const uint32_t own = S.cnt[par];
    uint64_t U = wave_max_u64(lane < W ? S.wmax[lane] : 0ull);  // this workgroup's best key

    // ---- 2. exchange --------------------------------------------------------
    // L lanes read one workgroup's header and its first L candidates at once, so most
    // candidates are here as soon as their header is; those beyond L follow.
    uint32_t C = own;
    if (G > 1) {
      const uint32_t capw = a.cap_wg;
      const uint32_t hp = G;  // pitch of one header word's array
      const size_t head = (size_t)kRoundsReplicas * kRoundsHeadWords * hp;
      const size_t cp = (size_t)G * capw;  // pitch of one word's array
      uint64_t *buf = f.xchg + (size_t)par * (head + NWC * cp);
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
          const uint64_t k = S.lk[q];
          const Rec<D> r = S.lc[q];
          uint64_t *w = cbuf + (size_t)g * capw + q;
          xchg_store(w, (k & 0xffffffff00000000ull) | e);
          xchg_store(w + cp, (k << 32) | e);
#pragma unroll
          for (int j = 0; j < D; ++j)
            xchg_store(w + (size_t)(2 + j) * cp,
                       ((uint64_t)(uint32_t)__float_as_int(r.c[j]) << 32) | e);
        }
      }
      const uint32_t L = G <= 128 ? 8 : 4;
      const uint32_t q = (uint32_t)tid / L;
      const uint32_t l = (uint32_t)tid & (L - 1);
      uint64_t w1 = 0, w2 = 0;
      if ((uint32_t)wave * 64 < G * L) {
        const uint64_t *h =
            buf + (size_t)(g % kRoundsReplicas) * kRoundsHeadWords * hp + q;
        const uint64_t *w = cbuf + (size_t)q * capw;
        uint32_t cq = 0;
        uint64_t v[NWC];
        const bool mine = q < G;
        bool here = false;  // candidate l of workgroup q is there
        if (mine) {
          const uint64_t deadline = now_ticks() + f.spin_ticks;
          for (;;) {
            const uint64_t w0 = xchg_load(h);
            w1 = xchg_load(h + hp);
            w2 = xchg_load(h + 2 * hp);
#pragma unroll
            for (uint32_t k = 0; k < NWC; ++k) v[k] = xchg_load(w + l + k * cp);
            bool all = true;
#pragma unroll
            for (uint32_t k = 0; k < NWC; ++k) all = all && (uint32_t)v[k] == e;
            cq = (uint32_t)(w0 >> 32);
            here = l < cq && cq <= capw;
            if ((uint32_t)w0 == e && (uint32_t)w1 == e && (uint32_t)w2 == e && (all || !here)) break;
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
            S.ck[at] = (v[0] & 0xffffffff00000000ull) | (v[1] >> 32);
            Rec<D> r;
#pragma unroll
            for (int j = 0; j < D; ++j) r.c[j] = __int_as_float((int)(v[2 + j] >> 32));
            S.cc[at] = r;
          }
          i += L;
          here = here && i < cq;
          if (here) {
            const uint64_t deadline = now_ticks() + f.spin_ticks;
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
      if (!__builtin_amdgcn_readfirstlane((int)S.ok)) {
        if (tid == 0) atomicOr(f.status, kStatusTimeout);
        return;
      }
      C = S.sum[par];
      const uint32_t got = S.at[par];
      if (got != C || C > (uint32_t)LIST) C = max(C, (uint32_t)LIST + 1);  // some did not fit
      if (C == 0) {
        // Nobody has a candidate: the best key of all is the exact bound.
        const uint64_t u = wave_max_u64((w1 & 0xffffffff00000000ull) | (w2 >> 32));
        if (lane == 0) S.wmax[wave] = (uint32_t)wave * 64 < G * L ? u : 0ull;
        lds_barrier();
        U = wave_max_u64(lane < W ? S.wmax[lane] : 0ull);
      }
    } else {
      if ((uint32_t)tid < own && tid < CAP) {
        S.ck[tid] = S.lk[tid];
        S.cc[tid] = S.lc[tid];
      }
      if (own > (uint32_t)CAP) C = max(own, (uint32_t)LIST + 1);
      lds_barrier();
    }
    if (tid == 0) {  // the other parity's counters: everybody has read them
      S.np = 0;
      S.cnt[par ^ 1] = 0;
      S.sum[par ^ 1] = 0;
      S.at[par ^ 1] = 0;
    }
    U = uniform_u64(U);
    C = (uint32_t)__builtin_amdgcn_readfirstlane((int)C);
    if (C > (uint32_t)LIST || C == 0) {
      // No picks: a smaller step, or the exact bound and a larger one.  From an exact bound
      // every step has a candidate, and halving ends at the best point alone, so a pick
      // comes within some 64 rounds; the count only guards the loop's end.
      np = 0;
      if (++idle > 1024) {
        if (tid == 0) atomicOr(f.status, kStatusTimeout);
        return;
      }
      if (C) {
        const uint64_t ns = (uint64_t)((double)step * sqrt((double)a.target / (double)C));
        step = ns < 1 ? 1 : ns;
      } else {
        T = U;
        if (Tg != ~0ull) step = step < ((uint64_t)1 << 60) ? step << 1 : step;
      }
      Tg = T > step ? T - step : 0;
      lds_barrier();
      continue;
    }

    // ---- 3. front -----------------------------------------------------------
    // Order of the candidates: how many keys exceed one's own, 16 at a time.
    {
      const uint32_t nc = (C + 63u) >> 6;
      const uint32_t nj = (C + 15u) >> 4;
      for (uint32_t job = wave; job < nc * nj; job += W) {
        const uint32_t jc = job / nc, ic = job - jc * nc;
        const uint32_t i = ic * 64 + lane;
        const uint64_t ki = S.ck[i];
        const uint64_t *kj = S.ck + jc * 16;
        uint32_t r = 0;
#pragma unroll 1
        for (int h = 0; h < 16; h += 8) {
#pragma unroll
          for (int l = 0; l < 8; ++l) r += kj[h + l] > ki ? 1u : 0u;
        }
        if (i < C && r) atomicAdd(&S.rank[i], r);
      }
    }
    lds_barrier();
    if ((uint32_t)tid < C) {
      const uint32_t r = S.rank[tid];
      if (r < (uint32_t)CAP) {
        S.sk[r] = S.ck[tid];
        S.sc[r] = S.cc[tid];
      } else if (r == (uint32_t)CAP) {
        S.te = S.ck[tid];  // the first one that the front does not see is the bound
      }
    }
    lds_barrier();
    const uint32_t F = min(C, (uint32_t)CAP);
    const uint32_t nc = (F + 63u) >> 6;
    // Which earlier candidates lower a candidate: bit j of candidate i's row, j < i, for the
    // sorted candidates.  A job is 64 candidates against 16 earlier ones.
    for (uint32_t job = wave, c = 0; c < nc;) {
      if (job >= 4 * (c + 1)) {
        job -= 4 * (c + 1);
        ++c;
        continue;
      }
      const uint32_t j0 = job * 16;
      if (j0 < F) {
        const uint32_t i = c * 64 + lane;
        const float v = __int_as_float((int)(uint32_t)(S.sk[i] >> 32) - 1);
        const Rec<D> ri = S.sc[i];
        float xi[D];
#pragma unroll
        for (int j = 0; j < D; ++j) xi[j] = ri.c[j];
        uint32_t bits = 0;
#pragma unroll 1
        for (int h = 12; h >= 0; h -= 4) {
#pragma unroll
          for (int l = 3; l >= 0; --l) {
            const Rec<D> rj = S.sc[j0 + h + l];
            float p[D];
#pragma unroll
            for (int j = 0; j < D; ++j) p[j] = rj.c[j];
            bits = bits + bits + (sqdist<D>(xi, p) < v ? 1u : 0u);
          }
        }
        S.low[job >> 1][i][job & 1] = (uint16_t)bits;
      }
      job += W;
    }
    lds_barrier();
    // The picks, were no candidate only partly lowered: each candidate that no earlier pick
    // lowers, settled in a few steps per 64 candidates rather than one by one.
    const uint32_t *rows = (const uint32_t *)&S.low[0][0][0];
    if (wave == 0) {
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
        if (lane == 0) S.acc[c] = acc[c];
      }
    }
    lds_barrier();
    // A candidate whose first lowering pick leaves its key above the bound raises the bound
    // to that key; a pick that does not lower itself ends the round.
    uint64_t key = 0;
    uint64_t taken = 0;
    Rec<D> ri;
    if ((uint32_t)wave < nc) {
      const uint32_t i = (uint32_t)tid;
      key = S.sk[i];
      ri = S.sc[i];
      const float v = __int_as_float((int)(uint32_t)(key >> 32) - 1);
      float xi[D];
#pragma unroll
      for (int j = 0; j < D; ++j) xi[j] = ri.c[j];
      taken = uniform_u64(S.acc[wave]);
      const bool mine = (taken >> lane) & 1;
      int by = -1;
#pragma unroll
      for (int w = CH - 1; w >= 0; --w) {
        if (w <= wave) {
          uint64_t k = ((uint64_t)rows[(2 * w + 1) * CAP + i] << 32) | rows[2 * w * CAP + i];
          if (w == wave) k &= ((uint64_t)1 << lane) - 1;
          k &= S.acc[w];
          if (k) by = w * 64 + __ffsll((unsigned long long)k) - 1;
        }
      }
      if (i < F && !mine && by >= 0) {
        const Rec<D> rb = S.sc[by];
        float p[D];
#pragma unroll
        for (int j = 0; j < D; ++j) p[j] = rb.c[j];
        const uint64_t nk = make_key(__float_as_int(sqdist<D>(xi, p)), (uint32_t)key);
        if (nk > Tg) atomicMax((unsigned long long *)&S.te, (unsigned long long)nk);
      }
      if (i < F && mine && !(sqdist<D>(xi, xi) < v)) atomicMin(&S.stop, i);
    }
    lds_barrier();
    T = uniform_u64(S.te);
    if ((uint32_t)wave < nc) {
      const uint32_t stop = S.stop;
      // Keys fall along the chunks: a chunk with picks has those before it whole.
      uint32_t at = 0;
      for (int w = 0; w < wave; ++w) at += (uint32_t)__popcll(S.acc[w]);
      taken &= __ballot(key > T && (uint32_t)tid <= stop);
      at = (uint32_t)__builtin_amdgcn_readfirstlane((int)at);
      const uint32_t room = a.s_end - s;
      if (taken) {
        const uint32_t q = at + lanes_below(taken);
        const uint32_t upto = min(at + (uint32_t)__popcll(taken), room);
        if (((taken >> lane) & 1) && q < room) {
          S.pt[q] = (uint32_t)key;
          S.pk[q] = ri;
          if (q == room - 1) S.last = key;
        }
        if (lane == 0) atomicMax(&S.np, upto);
        if (stop - (uint32_t)wave * 64 < 64u && ((taken >> (stop & 63u)) & 1) && lane == 0)
          S.stuck = 1;
      }
    }
    lds_barrier();
    idle = 0;
    np = (uint32_t)__builtin_amdgcn_readfirstlane((int)S.np);
    {
      // The square root damps the step against the count's own noise.
      double r = sqrt((double)a.target / (double)C);
      r = r > 4.0 ? 4.0 : r;
      const double ns = (double)step * r;
      step = ns < 1.0 ? 1 : (ns > 4.0e18 ? (uint64_t)1 << 61 : (uint64_t)ns);
      Tg = T > step ? T - step : 0;
    }
  }
}

template <int D, int P, int TIE>
__global__ void __launch_bounds__(kRoundsThreads) fps_rounds(RoundsParams a) {
  extern __shared__ uint64_t s_dyn[];
  __shared__ RoundsLds<D> S;
  rounds_cloud<D, P, TIE>(a, blockIdx.x, gridDim.x, S, s_dyn);
}

// A table entry in scalar registers: read in place, its fields would come through vector
// loads again after every store.
__device__ __forceinline__ RoundsParams uniform_params(const RoundsParams *p) {
  constexpr int N = sizeof(RoundsParams) / 4;
  union {
    RoundsParams a;
    uint32_t w[N];
  } u;
#pragma unroll
  for (int i = 0; i < N; ++i)
    u.w[i] = (uint32_t)__builtin_amdgcn_readfirstlane((int)((const uint32_t *)p)[i]);
  return u.a;
}

// Many clouds: workgroups claim member slots in order (or own one each), a job's members
// being consecutive slots.  A team's workgroups all claim before any waits for another: each
// claims its next slot only when done with the one before, so the first unfinished team is
// always complete or about to be.
template <int D, int P>
__global__ void __launch_bounds__(kRoundsThreads) fps_rounds_jobs(RoundsJobs j) {
  extern __shared__ uint64_t s_dyn[];
  __shared__ RoundsLds<D> S;
  __shared__ uint32_t s_slot;
  for (;;) {
    if (threadIdx.x == 0) s_slot = j.one_slot ? blockIdx.x : atomicAdd(j.claim, 1u);
    __syncthreads();
    const uint32_t slot = (uint32_t)__builtin_amdgcn_readfirstlane((int)s_slot);
    if (slot >= j.members) return;
    const RoundsParams a = uniform_params(
        j.table + (uint32_t)__builtin_amdgcn_readfirstlane((int)j.member_job[slot]));
    if (a.team > 1) {
      // Wait for the team to form, so that exchange waits are short ones.
      if (threadIdx.x == 0) {
        atomicAdd(a.ready, 1u);
        const uint64_t deadline = now_ticks() + j.team_ticks;
        uint32_t here = 1;
        while (__hip_atomic_load(a.ready, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) < a.team) {
          if (now_ticks() > deadline) {
            atomicOr(a.fps.status, kStatusTimeout);
            here = 0;
            break;
          }
          __builtin_amdgcn_s_sleep(1);
        }
        s_slot = here;
      }
      __syncthreads();
      if (!__builtin_amdgcn_readfirstlane((int)s_slot)) return;
    }
    rounds_cloud<D, P, kTieHighest>(
        a, (uint32_t)__builtin_amdgcn_readfirstlane((int)(slot - a.member_base)), a.team, S, s_dyn);
    if (j.one_slot) return;
    __syncthreads();
  }
}

#define ROUNDS(D, P)                                                                     \
  {D, kRoundsThreads, P, kTieHighest, (const void *)fps_rounds<D, P, kTieHighest>},      \
      {D, kRoundsThreads, P, kTieLowest, (const void *)fps_rounds<D, P, kTieLowest>}

static const KernelEntry kRounds[] = {
    ROUNDS(1, 4), ROUNDS(2, 1), ROUNDS(2, 4), ROUNDS(2, 8), ROUNDS(3, 1), ROUNDS(3, 4),
    ROUNDS(3, 8), ROUNDS(4, 1), ROUNDS(4, 4), ROUNDS(5, 1), ROUNDS(5, 4), ROUNDS(6, 1),
    ROUNDS(6, 4), ROUNDS(7, 1), ROUNDS(7, 4), ROUNDS(8, 1), ROUNDS(8, 4),
};

#define JOBS(D) {D, kRoundsThreads, 4, kTieHighest, (const void *)fps_rounds_jobs<D, 4>}

static const KernelEntry kJobs[] = {JOBS(1), JOBS(2), JOBS(3), JOBS(4)};

const KernelEntry *rounds_jobs_kernel(int dim) {
  return dim >= 1 && dim <= 4 ? &kJobs[dim - 1] : nullptr;
}

const KernelEntry *rounds_table(size_t *count) {
  *count = sizeof(kRounds) / sizeof(kRounds[0]);
  return kRounds;
}

}  // namespace fpsx
