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
// A cloud of 2^20 clustered points settles about 130 picks per round of 256 candidates.
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

// Inclusive prefix sum over the wave.
__device__ __forceinline__ uint32_t wave_scan_add(uint32_t v) {
  int x = (int)v;
#define STEP(ctrl, rm) x += __builtin_amdgcn_update_dpp(0, x, ctrl, rm, 0xf, false)
  STEP(0x111, 0xf);  // row_shr:1
  STEP(0x112, 0xf);  // row_shr:2
  STEP(0x114, 0xf);  // row_shr:4
  STEP(0x118, 0xf);  // row_shr:8
  STEP(0x142, 0xa);  // row_bcast:15
  STEP(0x143, 0xc);  // row_bcast:31
#undef STEP
  return (uint32_t)x;
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

template <int D, int P, int TIE>
__global__ void __launch_bounds__(kRoundsThreads) fps_rounds(RoundsParams a) {
  constexpr int W = kRoundsThreads / 64;
  constexpr int CAP = (int)kRoundsCap;
  constexpr int CH = CAP / 64;  // front waves
  constexpr uint32_t NWC = 2 + D;
  extern __shared__ uint64_t s_dyn[];  // best key of every block, then the boxes

  __shared__ uint64_t s_lk[CAP];      // this workgroup's candidates
  __shared__ float s_lc[D][CAP];
  __shared__ uint64_t s_ck[CAP];      // all candidates as they came
  __shared__ float s_cc[D][CAP];
  __shared__ uint64_t s_sk[CAP];      // sorted
  __shared__ float s_sc[D][CAP];
  __shared__ uint32_t s_rank[CAP];
  __shared__ uint32_t s_src[CAP];
  __shared__ float s_pk[D][CAP];      // picks of the round
  __shared__ uint32_t s_pt[CAP];      // their tie words
  __shared__ uint32_t s_cnt[2];     // candidates of this workgroup, by round parity
  __shared__ uint64_t s_wmax[W];
  __shared__ uint64_t s_wu[W];
  __shared__ uint32_t s_wtot[W];
  __shared__ uint32_t s_ok;
  __shared__ uint16_t s_low[CAP / 32][CAP][2];  // rows: which earlier candidates lower this one
  __shared__ uint64_t s_acc[CH];
  __shared__ uint64_t s_te;    // the bound that the round's picks exceed
  __shared__ uint32_t s_stop;  // first pick that does not lower itself
  __shared__ uint32_t s_np;
  __shared__ uint32_t s_stuck;

  const FpsParams &f = a.fps;
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const uint32_t G = gridDim.x;
  const uint32_t g = blockIdx.x;
  const uint32_t nbl = (a.nblocks - g + G - 1) / G;  // this workgroup's blocks: g, g + G, ...
  uint64_t *s_bkey = s_dyn;
  float *s_box = (float *)(s_dyn + nbl);  // [2 * D][nbl]

  if (tid == 0) {
    s_cnt[0] = 0;
    s_cnt[1] = 0;
    s_stuck = 0;
    s_ok = 1;
  }

  // Start: the forced picks, in pieces of CAP.
  uint32_t s = 0;        // picks recorded
  uint32_t np = 0;       // picks of the last round, in s_pk
  bool first = true;
  uint64_t T = ~0ull;    // every point's key is at most T
  uint64_t Tg = ~0ull;   // the round's bound
  uint64_t step = (uint64_t)1 << 51;  // a sixteenth of a binade
  uint32_t e = 0;        // rounds
  uint32_t idle = 0;     // rounds since the last pick

  for (;;) {
    // ---- forced picks -------------------------------------------------------
    const bool forced = s < f.n_starts;
    if (forced) {
      np = min(f.n_starts - s, (uint32_t)CAP);
      if ((uint32_t)tid < np) {
        uint64_t idx = f.starts[s + tid];
        if (idx >= f.n) {
          atomicOr(f.status, kStatusBadStart);
          idx = 0;
        }
#pragma unroll
        for (int j = 0; j < D; ++j) s_pk[j][tid] = f.pts[(size_t)idx * f.sp + (size_t)j * f.ld];
        s_pt[tid] = tie_of<TIE>((uint32_t)idx);
      }
      lds_barrier();
    }
    // ---- record -------------------------------------------------------------
    if (g == 0) {
      if ((uint32_t)tid < np) {
        f.out[s + tid] = tie_of<TIE>(s_pt[tid]);
        if (f.out_pts != nullptr) {
#pragma unroll
          for (int j = 0; j < D; ++j) f.out_pts[(size_t)(s + tid) * D + j] = s_pk[j][tid];
        }
      }
    }
    s += np;
    if (g == 0 && tid == 0) f.status[1] = e;
    if (s >= f.m) return;
    if (s_stuck) {
      // The last pick left its own key unchanged, so it stays the best for good.
      if (g == 0) {
        const uint32_t t = s_pt[np - 1];
        for (uint32_t q = s + tid; q < f.m; q += kRoundsThreads) {
          f.out[q] = tie_of<TIE>(t);
          if (f.out_pts != nullptr) {
#pragma unroll
            for (int j = 0; j < D; ++j) f.out_pts[(size_t)q * D + j] = s_pk[j][np - 1];
          }
        }
      }
      return;
    }
    const bool gather = s >= f.n_starts;  // no further forced picks
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
      bool any = first;
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
            float p[D];
#pragma unroll
            for (int j = 0; j < D; ++j) p[j] = s_pk[j][c * 64 + lane];
            const bool h = (uint32_t)(c * 64 + lane) < np && box_bound<D>(p, lo, hi) < bmax;
            hit[c] = __ballot(h);
            any = any || hit[c] != 0;
          }
        }
      }
      if (any || bkey > Tg) {
        float x[P][D], dm[P];
        uint32_t id[P];
#pragma unroll
        for (int k = 0; k < P; ++k) {
          const uint32_t p = base + (uint32_t)(k * 64 + lane);
          const uint32_t pc = min(p, f.n - 1);
#pragma unroll
          for (int j = 0; j < D; ++j)
            x[k][j] = a.pos[(size_t)pc * a.pos_sp + (size_t)j * a.pos_ld];
          id[k] = a.perm ? a.perm[pc] : pc;
          dm[k] = first ? f.init : f.dmin[pc];
        }
        if (base + 64 * P > f.n) {
#pragma unroll
          for (int k = 0; k < P; ++k)
            if (base + (uint32_t)(k * 64 + lane) >= f.n) dm[k] = -1.0f;
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
              float q[D];
#pragma unroll
              for (int j = 0; j < D; ++j) q[j] = s_pk[j][c * 64 + lane];
              do {
                const int l = __ffsll((unsigned long long)mm) - 1;
                mm &= mm - 1;
                float p[D];
#pragma unroll
                for (int j = 0; j < D; ++j) p[j] = readlane_f(q[j], l);
#pragma unroll
                for (int k = 0; k < P; ++k) dm[k] = min_keep(sqdist<D>(x[k], p), dm[k]);
              } while (mm);
            }
          }
#pragma unroll
          for (int k = 0; k < P; ++k) {
            const uint32_t p = base + (uint32_t)(k * 64 + lane);
            if (p < f.n) f.dmin[p] = dm[k];
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
          if (lane == 0) at = atomicAdd(&s_cnt[(e + 1) & 1], total);
          at = (uint32_t)__builtin_amdgcn_readfirstlane((int)at);
#pragma unroll
          for (int k = 0; k < P; ++k) {
            const uint32_t q = at + lanes_below(m[k]);
            if (((m[k] >> lane) & 1) && q < (uint32_t)CAP) {
              s_lk[q] = make_key(__float_as_int(dm[k]), tie_of<TIE>(id[k]));
#pragma unroll
              for (int j = 0; j < D; ++j) s_lc[j][q] = x[k][j];
            }
            at += (uint32_t)__popcll(m[k]);
          }
        }
      }
      wmax = bkey > wmax ? bkey : wmax;
    }
    first = false;
    if (!gather) {
      lds_barrier();
      continue;
    }
    if (lane == 0) s_wmax[wave] = wmax;
    lds_barrier();
    ++e;
    uint32_t C = s_cnt[e & 1];
    uint64_t U = wave_max_u64(lane < W ? s_wmax[lane] : 0ull);  // this workgroup's best key

    // ---- 2. exchange --------------------------------------------------------
    bool over;
    if (G > 1) {
      const uint32_t capw = a.cap_wg;
      over = C > capw;
      const size_t head = (size_t)kRoundsReplicas * kRoundsHeadWords * kRoundsMaxGrid;
      const size_t cands = (size_t)NWC * G * capw;
      uint64_t *buf = f.xchg + (size_t)(e & 1u) * (head + cands);
      uint64_t *cbuf = buf + head;
      const size_t cp = (size_t)G * capw;  // pitch of one word's array
      if (wave == 0) {
        if (lane < (int)(kRoundsReplicas * kRoundsHeadWords)) {
          const uint32_t rep = (uint32_t)lane / kRoundsHeadWords;
          const uint32_t k = (uint32_t)lane - rep * kRoundsHeadWords;
          const uint32_t v = k == 0 ? (C | (over ? 0x80000000u : 0u))
                                    : (k == 1 ? (uint32_t)(U >> 32) : (uint32_t)U);
          xchg_store(buf + ((size_t)rep * kRoundsHeadWords + k) * kRoundsMaxGrid + g,
                     ((uint64_t)v << 32) | e);
        }
      } else if (!over) {
        for (uint32_t q = (uint32_t)tid - 64; q < C; q += kRoundsThreads - 64) {
          const uint64_t k = s_lk[q];
          uint64_t *w = cbuf + (size_t)g * capw + q;
          xchg_store(w, (k & 0xffffffff00000000ull) | e);
          xchg_store(w + cp, (k << 32) | e);
#pragma unroll
          for (int j = 0; j < D; ++j)
            xchg_store(w + (size_t)(2 + j) * cp,
                       ((uint64_t)(uint32_t)__float_as_int(s_lc[j][q]) << 32) | e);
        }
      }
      const uint32_t PW = (G + 63u) >> 6;
      uint32_t cq = 0;
      uint32_t incl = 0;
      if ((uint32_t)wave < PW) {
        const uint32_t q = (uint32_t)tid;
        const uint64_t *h = buf + (size_t)(g % kRoundsReplicas) * kRoundsHeadWords * kRoundsMaxGrid + q;
        uint64_t w0 = 0, w1 = 0, w2 = 0;
        bool ok = true;
        if (q < G) {
          const uint64_t deadline = now_ticks() + f.spin_ticks;
          for (;;) {
            w0 = xchg_load(h);
            w1 = xchg_load(h + kRoundsMaxGrid);
            w2 = xchg_load(h + 2 * kRoundsMaxGrid);
            if ((uint32_t)w0 == e && (uint32_t)w1 == e && (uint32_t)w2 == e) break;
            if (now_ticks() > deadline) {
              ok = false;
              break;
            }
          }
        }
        const bool wave_ok = __ballot(!ok) == 0;
        cq = (uint32_t)(w0 >> 32);
        const bool ov = __ballot((cq & 0x80000000u) != 0) != 0;
        cq &= 0x7fffffffu;
        incl = wave_scan_add(cq);
        const uint64_t u = wave_max_u64((w1 & 0xffffffff00000000ull) | (w2 >> 32));
        if (lane == 63) {
          s_wtot[wave] = (incl & 0x7fffffffu) | (ov ? 0x80000000u : 0u);
          s_wu[wave] = u;
          if (!wave_ok) s_ok = 0;
        }
        if (PW == 1 && !ov) {
          const uint32_t off = incl - cq;
          for (uint32_t i = 0; i < cq && off + i < (uint32_t)CAP; ++i) s_src[off + i] = q * capw + i;
        }
      }
      lds_barrier();
      if (!s_ok) {
        if (tid == 0) atomicOr(f.status, kStatusTimeout);
        return;
      }
      C = 0;
      over = false;
      U = 0;
      uint32_t before = 0;
      for (uint32_t w = 0; w < PW; ++w) {
        const uint32_t t = s_wtot[w];
        if (w < (uint32_t)wave) before += t & 0x7fffffffu;
        C += t & 0x7fffffffu;
        over = over || (t & 0x80000000u);
        U = s_wu[w] > U ? s_wu[w] : U;
      }
      over = over || C > (uint32_t)CAP;
      if (PW > 1 && !over) {
        if ((uint32_t)wave < PW) {
          const uint32_t off = before + incl - cq;
          for (uint32_t i = 0; i < cq; ++i) s_src[off + i] = (uint32_t)tid * capw + i;
        }
        lds_barrier();
      }
      if (!over && (uint32_t)tid < C) {
        const uint64_t *w = cbuf + s_src[tid];
        uint64_t v[NWC];
        const uint64_t deadline = now_ticks() + f.spin_ticks;
        for (;;) {
          bool all = true;
#pragma unroll
          for (uint32_t k = 0; k < NWC; ++k) v[k] = xchg_load(w + k * cp);
#pragma unroll
          for (uint32_t k = 0; k < NWC; ++k) all = all && (uint32_t)v[k] == e;
          if (all) break;
          if (now_ticks() > deadline) {
            s_ok = 0;
            break;
          }
        }
        s_ck[tid] = (v[0] & 0xffffffff00000000ull) | (v[1] >> 32);
#pragma unroll
        for (int j = 0; j < D; ++j) s_cc[j][tid] = __int_as_float((int)(v[2 + j] >> 32));
      }
    } else {
      over = C > (uint32_t)CAP;
      if (!over && (uint32_t)tid < C) {
        s_ck[tid] = s_lk[tid];
#pragma unroll
        for (int j = 0; j < D; ++j) s_cc[j][tid] = s_lc[j][tid];
      }
    }
    if (tid < CAP) s_rank[tid] = 0;
    if (tid == 0) {
      s_cnt[(e + 1) & 1] = 0;  // read by everybody before this round's first barrier
      s_te = Tg;
      s_stop = ~0u;
    }
    lds_barrier();
    if (!s_ok) {
      if (tid == 0) atomicOr(f.status, kStatusTimeout);
      return;
    }
    U = uniform_u64(U);
    C = (uint32_t)__builtin_amdgcn_readfirstlane((int)C);
    if (over || C == 0) {
      // No picks: a smaller step, or the exact bound and a larger one.  From an exact bound
      // every step has a candidate, and halving ends at the best point alone, so a pick
      // comes within some 64 rounds; the count only guards the loop's end.
      np = 0;
      if (++idle > 1024) {
        if (tid == 0) atomicOr(f.status, kStatusTimeout);
        return;
      }
      if (over) {
        const double r = sqrt((double)a.target / (double)(C > 2 * a.target ? C : 2 * a.target));
        const uint64_t ns = (uint64_t)((double)step * r);
        step = ns < 1 ? 1 : ns;
      } else {
        T = U;
        if (Tg != ~0ull) step = step < ((uint64_t)1 << 60) ? step << 1 : step;
      }
      Tg = T > step ? T - step : 0;
      continue;
    }

    // ---- 3. front -----------------------------------------------------------
    const uint32_t nc = (C + 63u) >> 6;
    for (uint32_t job = wave; job < nc * nc; job += W) {
      const uint32_t ic = job % nc, jc = job / nc;
      const uint32_t i = ic * 64 + lane;
      const uint64_t ki = i < C ? s_ck[i] : ~0ull;
      const uint32_t jl = jc * 64 + lane;
      const uint64_t kj = jl < C ? s_ck[jl] : 0ull;
      const int jn = (int)min(64u, C - jc * 64);
      uint32_t r = 0;
      for (int l = 0; l < jn; ++l) r += readlane_u64(kj, l) > ki ? 1u : 0u;
      if (i < C) atomicAdd(&s_rank[i], r);
    }
    lds_barrier();
    if ((uint32_t)tid < C) {
      const uint32_t r = s_rank[tid];
      s_sk[r] = s_ck[tid];
#pragma unroll
      for (int j = 0; j < D; ++j) s_sc[j][r] = s_cc[j][tid];
    }
    lds_barrier();
    // Which earlier candidates lower a candidate: bit j of candidate i's row, j < i, for the
    // sorted candidates.  A job is 64 candidates against 16 earlier ones.
    for (uint32_t job = wave, c = 0; c < nc;) {
      if (job >= 4 * (c + 1)) {
        job -= 4 * (c + 1);
        ++c;
        continue;
      }
      const uint32_t j0 = job * 16;
      if (j0 < C) {
        const uint32_t i = c * 64 + lane;
        const float v = __int_as_float((int)(uint32_t)(s_sk[i] >> 32) - 1);
        float x[D], q[D];
#pragma unroll
        for (int j = 0; j < D; ++j) {
          x[j] = s_sc[j][i];
          q[j] = s_sc[j][j0 + (lane & 15)];
        }
        uint32_t bits = 0;
#pragma unroll
        for (int l = 15; l >= 0; --l) {
          float p[D];
#pragma unroll
          for (int j = 0; j < D; ++j) p[j] = readlane_f(q[j], l);
          bits = bits + bits + (sqdist<D>(x, p) < v ? 1u : 0u);
        }
        s_low[job >> 1][i][job & 1] = (uint16_t)bits;
      }
      job += W;
    }
    lds_barrier();
    // The picks, were no candidate only partly lowered: each candidate that no earlier pick
    // lowers, settled in a few steps per 64 candidates rather than one by one.
    if (wave == 0) {
      uint64_t low[CH][CH];
#pragma unroll
      for (int c = 0; c < CH; ++c)
#pragma unroll
        for (int w = 0; w <= c; ++w) {
          const uint32_t *r = (const uint32_t *)&s_low[0][0][0];
          low[c][w] = ((uint64_t)r[(2 * w + 1) * CAP + c * 64 + lane] << 32) |
                      r[2 * w * CAP + c * 64 + lane];
        }
      uint64_t acc[CH];
#pragma unroll
      for (int c = 0; c < CH; ++c) {
        acc[c] = 0;
        if ((uint32_t)c < nc) {
          uint64_t hitc = 0;
#pragma unroll
          for (int w = 0; w < c; ++w) hitc |= low[c][w] & acc[w];
          const uint64_t own = low[c][c] & (((uint64_t)1 << lane) - 1);
          uint64_t open = __ballot((uint32_t)(c * 64 + lane) < C && hitc == 0);
          while (open) {
            const uint64_t free = __ballot((own & open) == 0) & open;
            acc[c] |= free;
            open &= ~free;
            open &= ~__ballot((own & free) != 0);
          }
        }
        if (lane == 0) s_acc[c] = acc[c];
      }
    }
    lds_barrier();
    // A candidate whose first lowering pick leaves its key above the bound raises the bound
    // to that key; a pick that does not lower itself ends the round.
    if ((uint32_t)wave < nc) {
      const uint32_t i = (uint32_t)tid;
      const uint64_t key = s_sk[i];
      const float v = __int_as_float((int)(uint32_t)(key >> 32) - 1);
      float x[D];
#pragma unroll
      for (int j = 0; j < D; ++j) x[j] = s_sc[j][i];
      const uint64_t mine = uniform_u64(s_acc[wave]);
      const bool taken = (mine >> lane) & 1;
      int by = -1;
#pragma unroll
      for (int w = CH - 1; w >= 0; --w) {
        if (w <= wave) {
          const uint32_t *r = (const uint32_t *)&s_low[0][0][0];
          uint64_t k = ((uint64_t)r[(2 * w + 1) * CAP + i] << 32) | r[2 * w * CAP + i];
          if (w == wave) k &= ((uint64_t)1 << lane) - 1;
          k &= s_acc[w];
          if (k) by = w * 64 + __ffsll((unsigned long long)k) - 1;
        }
      }
      if (i < C && !taken && by >= 0) {
        float p[D];
#pragma unroll
        for (int j = 0; j < D; ++j) p[j] = s_sc[j][by];
        const uint64_t nk = make_key(__float_as_int(sqdist<D>(x, p)), (uint32_t)key);
        if (nk > Tg) atomicMax((unsigned long long *)&s_te, (unsigned long long)nk);
      }
      if (i < C && taken && !(sqdist<D>(x, x) < v)) atomicMin(&s_stop, i);
    }
    lds_barrier();
    T = uniform_u64(s_te);
    const uint32_t stop = (uint32_t)__builtin_amdgcn_readfirstlane((int)s_stop);
    if ((uint32_t)wave < nc) {
      uint32_t at = 0;
      uint64_t mine = 0;
      for (uint32_t c = 0; c < nc; ++c) {
        const uint32_t i = c * 64 + lane;
        const uint64_t m =
            __ballot(i < C && s_sk[i] > T && i <= stop) & uniform_u64(s_acc[c]);
        if (c < (uint32_t)wave) at += (uint32_t)__popcll(m);
        if (c == (uint32_t)wave) mine = m;
      }
      const uint32_t room = f.m - s;
      const uint32_t q = at + lanes_below(mine);
      if (((mine >> lane) & 1) && q < room) {
        s_pt[q] = (uint32_t)s_sk[tid];
#pragma unroll
        for (int j = 0; j < D; ++j) s_pk[j][q] = s_sc[j][tid];
      }
      if ((uint32_t)wave == nc - 1 && lane == 0) {
        const uint32_t all = at + (uint32_t)__popcll(mine);
        s_np = all < room ? all : room;
        if (stop < C && s_sk[stop] > T) s_stuck = 1;
      }
    }
    lds_barrier();
    idle = 0;
    np = (uint32_t)__builtin_amdgcn_readfirstlane((int)s_np);
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

#define ROUNDS(D, P)                                                                     \
  {D, kRoundsThreads, P, kTieHighest, (const void *)fps_rounds<D, P, kTieHighest>},      \
      {D, kRoundsThreads, P, kTieLowest, (const void *)fps_rounds<D, P, kTieLowest>}

static const KernelEntry kRounds[] = {ROUNDS(3, 1), ROUNDS(3, 4), ROUNDS(3, 8)};

const KernelEntry *rounds_table(size_t *count) {
  *count = sizeof(kRounds) / sizeof(kRounds[0]);
  return kRounds;
}

}  // namespace fpsx
