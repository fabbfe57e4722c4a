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
// workgroups: 165 rounds of 11.6 us, the paired pass kernel 8203 exchanges of 3.4 us).  Of a
// round (50 K points, 64 workgroups, 64 rounds of 9.7 us): update 2.2 us with the wait for the
// slowest wave, exchange 3.0, sorting 0.9, rows 1.4, settling 0.4, the bound and the picks 0.6.
// Settling the candidates one by one instead took 450 ns a pick.  A block per wave in
// registers, the candidates loaded beside the headers and the best 256 taken from up to 512
// brought 2^20 clustered points from 2.67 to 2.13 ms, 100 K / 50 K picks from 4.52 to 3.44 ms;
// jobs of half-waves in the sorting and the rows and one pass for bound and picks, 50 K / 4096
// picks from 668 to 654 us, 2^22 / 4096 picks 2.09 to 2.03 ms.  Deciding the candidates that a
// cut leaves in a further pass saves one round in ten to five, and costs as much.
#include "fps_rounds.hpp"

#include "fps_device.hpp"
#include "fps_kernels.hpp"
#include "fps_rounds_device.hpp"

namespace fpsx {

// LDS of a workgroup beside its blocks' boxes and best keys.
template <int D>
struct RoundsLds : RoundsCounts {
  static constexpr int CAP = (int)kRoundsCap;    // candidates the front decides on
  static constexpr int LIST = (int)kRoundsList;  // candidates that may come in
  static constexpr int W = kRoundsThreads / 64;
  alignas(16) uint64_t ck[LIST];  // candidates as they came
  Rec<D> cc[LIST];
  Rec<D> pk[CAP];                 // picks of the round
  uint32_t pt[CAP];               // their keys' low halves: tie words
  uint32_t pv[CAP];               // and high halves
  uint32_t rank[LIST];
  uint64_t sk[CAP];               // sorted candidates
  Rec<D> sc[CAP];
  uint16_t low[CAP / 32][CAP][2];  // rows: which earlier candidates lower this one
  uint64_t lk[CAP];                // this workgroup's candidates
  Rec<D> lc[CAP];
  uint64_t acc[CAP / 64];
};

// Workgroup `group` of G working on one cloud: picks a.s_begin .. a.s_end - 1.
template <int D, int P, int TIE>
__device__ __forceinline__ void rounds_cloud(ParamsPtr params, const uint32_t group,
                                             const uint32_t G, RoundsLds<D> &S, uint64_t *s_dyn) {
  constexpr int W = RoundsLds<D>::W;
  constexpr int CAP = RoundsLds<D>::CAP;
  constexpr int LIST = RoundsLds<D>::LIST;
  constexpr int CH = CAP / 64;
  int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const uint32_t s_begin = params->s_begin;
  const uint32_t nbl = (params->nblocks - group + G - 1) / G;  // blocks group, group + G, ...
  const bool resident = nbl <= (uint32_t)W;          // a block per wave stays in registers
  uint64_t *s_bkey = s_dyn;
  float *s_box = (float *)(s_dyn + nbl);  // [2 * D][nbl]

  if (tid == 0) {
    S.last = ~0ull;
    S.clear(0);
    S.clear(1);
    S.stuck = 0;
    S.ok = 1;
  }

  if (s_begin) lds_barrier();  // (a fresh run has one after its forced picks)

  uint32_t s = s_begin;    // picks recorded
  uint32_t np = 0;         // picks of the last round, in S.pk
  uint32_t fresh = 1;      // the blocks have not been read yet
  uint64_t T = ~0ull;    // every point's key is at most T
  uint64_t Tg = ~0ull;   // the round's bound
  uint64_t step = (uint64_t)1 << 51;  // a sixteenth of a binade
  if (s_begin) {
    // A run taken up again: no key exceeds that of its last pick.
    const uint32_t *carry = params->carry;
    T = uniform_u64(((uint64_t)carry[0] << 32) | carry[1]);
    step = uniform_u64(((uint64_t)carry[2] << 32) | carry[3]);
    Tg = round_bound(T, step);
  }
  uint32_t e = 0;        // rounds
  uint32_t empty = 0;    // the last round had no candidate
  float x[P][D], dm[P];  // the block in hand
  uint32_t id[P];

  for (;;) {
    // Rewritten each round: addresses formed from them would otherwise be kept in registers
    // over the whole loop, beside the block.
    asm volatile("" : "+v"(tid), "+s"(params));
    const __attribute__((address_space(4))) RoundsParams &a = *params;
    const __attribute__((address_space(4))) FpsParams &f = a.fps;
    uint32_t g = (uint32_t)__builtin_amdgcn_readfirstlane((int)group);
    asm volatile("" : "+s"(g));
    const int lane = tid & 63;
    // What the rounds carry is the same in every lane, which the compiler cannot see through
    // the loop's several exits; in vector registers its branches would run under masks (the
    // update loop a fifth slower).
    s = uniform_u32(s);
    np = uniform_u32(np);
    e = uniform_u32(e);
    empty = uniform_u32(empty);
    T = uniform_u64(T);
    Tg = uniform_u64(Tg);
    step = uniform_u64(step);
    const bool first = uniform_u32(fresh) != 0;
    // ---- forced picks, in pieces of CAP -------------------------------------
    if (s < f.n_starts) {
      np = min(f.n_starts - s, (uint32_t)CAP);
      if ((uint32_t)tid < np) {
        uint64_t idx = f.starts ? f.starts[s + tid] : a.start;
        if (idx >= f.n) {
          rounds_fail(params, kStatusBadStart);
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
    const bool cut = s >= a.s_end;
    // (a last pick that left its own key unchanged stays the best for good)
    const bool stuck = uniform_u32(!cut && np && S.stuck) != 0;
    if (stuck && g == 0) {
      const uint32_t t = S.pt[np - 1];
      for (uint32_t q = s + tid; q < a.s_end; q += kRoundsThreads) {
        f.out[q] = tie_of<TIE>(t);
        if (f.out_pts != nullptr) {
#pragma unroll
          for (int j = 0; j < D; ++j) f.out_pts[(size_t)q * D + j] = S.pk[np - 1].c[j];
        }
      }
    }
    if (stuck && a.s_end >= f.m) return;
    // The picks of this part are made: apply them and save.
    const bool last = cut || stuck;
    if (last && g == 0 && tid == 0) {
      a.carry[0] = cut ? (uint32_t)(S.last >> 32) : ~0u;
      a.carry[1] = cut ? (uint32_t)S.last : ~0u;
      a.carry[2] = (uint32_t)(step >> 32);
      a.carry[3] = (uint32_t)step;
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
          // Every load of the block before any use: one memory round trip (chosen per point, the
          // kind of load made one trip of each: 2^24 points, 2048 picks, 4.84 against 4.58 ms;
          // 256 clouds of 2 K to 65 K points 3.72 against 3.24 ms).
          uint32_t pc[P];
#pragma unroll
          for (int k = 0; k < P; ++k) pc[k] = min(base + (uint32_t)(k * 64 + lane), f.n - 1);
          if (first && s_begin == 0) {
#pragma unroll
            for (int k = 0; k < P; ++k) dm[k] = f.init;
          } else {
#pragma unroll
            for (int k = 0; k < P; ++k) dm[k] = f.dmin[pc[k]];
          }
          if (a.rec) {
#pragma unroll
            for (int k = 0; k < P; ++k) {
              const float4 r = a.rec[pc[k]];
              const float r3[3] = {r.x, r.y, r.z};
#pragma unroll
              for (int j = 0; j < D; ++j)
                x[k][j] = j < 3 ? r3[j < 3 ? j : 0] : a.rest[(size_t)(j - 3) * f.n + pc[k]];
              id[k] = (uint32_t)__float_as_int(r.w);
            }
          } else {
#pragma unroll
            for (int k = 0; k < P; ++k) {
#pragma unroll
              for (int j = 0; j < D; ++j)
                x[k][j] = f.pts[(size_t)pc[k] * f.sp + (size_t)j * f.ld];
              id[k] = pc[k];
            }
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
        bkey = uniform_u64(bkey);
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
      wmax = uniform_u64(bkey > wmax ? bkey : wmax);
    }
    fresh = 0;
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
    lds_barrier();
    ++e;
    const uint32_t par = e & 1u;
    const uint32_t own = S.cnt[par];
    uint64_t U = wave_max_u64(lane < W ? S.wmax[lane] : 0ull);  // this workgroup's best key

    // ---- 2. exchange --------------------------------------------------------
    uint32_t C = own;
    if (G > 1) {
      if (!rounds_exchange<D, LIST>(f.xchg, e == 1 ? a.form_ticks : f.spin_ticks, a.cap_wg, G, g,
                                    e, tid, wave, S, S.lk, S.lc, S.ck, S.cc, C, U)) {
        if (tid == 0) rounds_fail(params, kStatusTimeout);
        return;
      }
    } else {
      if ((uint32_t)tid < own && tid < CAP) {
        S.ck[tid] = S.lk[tid];
        S.cc[tid] = S.lc[tid];
      }
      if (own > (uint32_t)CAP) C = max(own, (uint32_t)LIST + 1);
      lds_barrier();
    }
    if (tid == 0) S.clear(par ^ 1);  // everybody has read the last round's
    U = uniform_u64(U);
    C = (uint32_t)__builtin_amdgcn_readfirstlane((int)C);
    if (C > (uint32_t)LIST || C == 0) {
      // Too many candidates, or none: the best point of all is the pick, and the exact bound.
      // (Without that pick a point held many times over took a round or two for each copy's
      // step: 4096 points, half of them one point, 192 picks 643 us, so 195, by passes 237.)
      if (tid == 0) {
        const size_t idx = tie_of<TIE>((uint32_t)U);
        float x0[D];
        Rec<D> r;
#pragma unroll
        for (int j = 0; j < D; ++j) r.c[j] = x0[j] = f.pts[idx * f.sp + (size_t)j * f.ld];
        S.pk[0] = r;
        S.pt[0] = (uint32_t)U;
        if (!(sqdist<D>(x0, x0) < __int_as_float((int)(uint32_t)(U >> 32) - 1))) S.stuck = 1;
        S.last = U;
      }
      np = 1;
      if (C)
        step = less_step(step, a.target, C);
      else if (empty)
        step = next_step(step, a.target, 1);
      empty = C == 0;
      T = U;
      Tg = round_bound(T, step);
      lds_barrier();
      continue;
    }

    // ---- 3. front -----------------------------------------------------------
    rank_candidates(S.ck, S.rank, C, tid, wave);
    lds_barrier();
    if ((uint32_t)tid < C) {
      const uint32_t r = S.rank[tid];
      if (r < (uint32_t)CAP) {
        S.sk[r] = S.ck[tid];
        S.sc[r] = S.cc[tid];
      } else if (r == (uint32_t)CAP) {
        S.te[par] = S.ck[tid];  // the first one that the front does not see is the bound
      }
    }
    lds_barrier();
    const uint32_t F = min(C, (uint32_t)CAP);
    const uint32_t nc = (F + 63u) >> 6;
    // Which earlier candidates lower a candidate: bit j of candidate i's row, j < i, for the
    // sorted candidates.  A job is 32 candidates against 32 earlier ones, 16 for each half of
    // the wave: the triangle and its ragged end then waste few lanes (146 candidates: 15 jobs,
    // one a wave, against 22 of 64 x 16: 1.3 us a round against 1.65).
    for (uint32_t job = wave, c = 0; c * 32 < F;) {
      if (job > c) {
        job -= c + 1;
        ++c;
        continue;
      }
      const uint32_t i = c * 32 + (lane & 31);
      const uint32_t jb = job * 2 + (lane >> 5);  // block of 16 earlier ones
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
          const Rec<D> rj = S.sc[jb * 16 + h + l];
          float p[D];
#pragma unroll
          for (int j = 0; j < D; ++j) p[j] = rj.c[j];
          bits = bits + bits + (sqdist<D>(xi, p) < v ? 1u : 0u);
        }
      }
      S.low[job][i][lane >> 5] = (uint16_t)bits;
      job += W;
    }
    lds_barrier();
    const uint32_t *rows = (const uint32_t *)&S.low[0][0][0];
    if (wave == 0) settle_candidates<CAP>(rows, F, lane, S.acc);
    if (wave == 1 && lane == 0) S.step = next_step(step, a.target, C);  // (in its shadow)
    lds_barrier();
    // The picks, in order.  A candidate whose first lowering pick leaves its key above the
    // bound raises the bound to that key, and a pick that does not lower itself ends the round:
    // both are rare and cut the picks below.
    if ((uint32_t)wave < nc) {
      const uint32_t i = (uint32_t)tid;
      const uint64_t key = S.sk[i];
      const Rec<D> ri = S.sc[i];
      const float v = __int_as_float((int)(uint32_t)(key >> 32) - 1);
      float xi[D];
#pragma unroll
      for (int j = 0; j < D; ++j) xi[j] = ri.c[j];
      uint64_t acc[CH];
      uint32_t at = 0, all = 0;
#pragma unroll
      for (int w = 0; w < CH; ++w) {
        acc[w] = uniform_u64(S.acc[w]);
        if (w < wave) at += (uint32_t)__popcll(acc[w]);
        all += (uint32_t)__popcll(acc[w]);
      }
      const uint64_t taken = uniform_u64(S.acc[wave]);
      const bool mine = (taken >> lane) & 1;
      int by = -1;
#pragma unroll
      for (int w = CH - 1; w >= 0; --w) {
        if (w <= wave) {
          uint64_t k = ((uint64_t)rows[(2 * w + 1) * CAP + i] << 32) | rows[2 * w * CAP + i];
          if (w == wave) k &= ((uint64_t)1 << lane) - 1;
          k &= acc[w];
          if (k) by = w * 64 + __ffsll((unsigned long long)k) - 1;
        }
      }
      const uint32_t q = at + lanes_below(taken);
      if (mine) {
        S.pt[q] = (uint32_t)key;
        S.pv[q] = (uint32_t)(key >> 32);
        S.pk[q] = ri;
        if (!(sqdist<D>(xi, xi) < v)) atomicMin(&S.stop[par], q);
      } else if (i < F && by >= 0) {
        const Rec<D> rb = S.sc[by];
        float p[D];
#pragma unroll
        for (int j = 0; j < D; ++j) p[j] = rb.c[j];
        const float d = sqdist<D>(xi, p);
        const uint64_t nk = make_key(__float_as_int(d), (uint32_t)key);
        if (nk > Tg) atomicMax((unsigned long long *)&S.te[par], (unsigned long long)nk);
      }
      if (tid == 0) S.np[par] = all;
    }
    lds_barrier();
    np = uniform_u32(S.np[par]);
    T = uniform_u64(S.te[par]);
    T = T > Tg ? T : Tg;
    const uint32_t stop = uniform_u32(S.stop[par]);
    if (T > Tg || stop < np) {
      // Picks up to the stop whose keys exceed the bound (keys fall along the picks).
      uint32_t keep = 0;
      for (uint32_t c = 0; c < np; c += 64) {
        const uint32_t q = c + lane;
        const uint64_t k = q < np ? ((uint64_t)S.pv[q] << 32) | S.pt[q] : 0ull;
        keep += (uint32_t)__popcll(__ballot(k > T && q <= stop));
      }
      np = keep;
      if (stop < np) {
        lds_barrier();  // (nobody reads S.stuck between)
        if (tid == 0) S.stuck = 1;
        lds_barrier();
      }
    }
    np = min(np, a.s_end - s);
    if (s + np == a.s_end && a.s_end < f.m && tid == 0)
      S.last = ((uint64_t)S.pv[np - 1] << 32) | S.pt[np - 1];
    empty = 0;
    step = uniform_u64(S.step);
    Tg = round_bound(T, step);
  }
}

template <int D, int P, int TIE>
__global__ void __launch_bounds__(kRoundsThreads) fps_rounds(RoundsParams) {
  extern __shared__ uint64_t s_dyn[];
  __shared__ RoundsLds<D> S;
  // (its only argument)
  rounds_cloud<D, P, TIE>((ParamsPtr)__builtin_amdgcn_kernarg_segment_ptr(), blockIdx.x, gridDim.x,
                          S, s_dyn);
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
  __shared__ uint32_t s_here;  // (a word of its own: waves read s_slot while it is written)
  for (;;) {
    if (threadIdx.x == 0) s_slot = j.one_slot ? blockIdx.x : atomicAdd(j.claim, 1u);
    __syncthreads();
    const uint32_t slot = (uint32_t)__builtin_amdgcn_readfirstlane((int)s_slot);
    if (slot >= j.members) return;
    const ParamsPtr p = (ParamsPtr)j.table + uniform_u32(j.member_job[slot]);
    if (p->team > 1 && !j.one_slot) {
      // Wait for the team to form, so that exchange waits are short ones.  (With a slot each, a
      // team's workgroups start together, and the first exchange finds out.)
      if (threadIdx.x == 0) {
        atomicAdd(p->ready, 1u);
        const uint64_t deadline = now_ticks() + j.team_ticks;
        s_here = 1;
        while (__hip_atomic_load(p->ready, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) < p->team) {
          if (now_ticks() > deadline) {
            rounds_fail(p, kStatusTimeout);
            s_here = 0;
            break;
          }
          __builtin_amdgcn_s_sleep(1);
        }
      }
      __syncthreads();
      if (!__builtin_amdgcn_readfirstlane((int)s_here)) return;
    }
    rounds_cloud<D, P, kTieHighest>(p, uniform_u32(slot - p->member_base), p->team, S, s_dyn);
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
