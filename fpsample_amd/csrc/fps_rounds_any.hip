// fps_rounds_any.hip -- threshold rounds (fps_rounds.hip) in any dimension.
//
// Beyond eight dimensions a point's coordinates do not fit a lane's registers, and a spatial
// order prunes nothing.  So a round's picks go to every point: a wave takes 64 points and eight
// picks, reads each coordinate of the points once (arrays by coordinate, 256 bytes a load) and
// subtracts the eight picks' coordinates from LDS; several waves share a block, their minima
// meeting in LDS.  Candidates are exchanged by key alone, and the coordinates of the best kAnyCap
// are read by index once they are sorted.
//
// What bounds it: the vector ALUs, in the update (three operations per point, pick and
// coordinate) and in the candidates' rows.  20000 points of 32 dimensions, 2000 picks: the
// one-pick streaming kernel takes 5.2 us a pick, this one 0.39 (49 rounds of 16 us).
#include "fps_device.hpp"
#include "fps_rounds.hpp"
#include "fps_rounds_device.hpp"

namespace fpsx {

namespace {

constexpr int kGroup = 8;  // picks of one job

// Squared distances of this lane's point to kGroup rows of LDS, summed in dimension order.
// x(j) gives coordinate j of the point.
template <class X>
__device__ __forceinline__ void group_dist(X x, const float *const (&row)[kGroup], uint32_t dim,
                                           float (&acc)[kGroup]) {
#pragma unroll
  for (int l = 0; l < kGroup; ++l) acc[l] = 0.0f;
  uint32_t j = 0;
  for (; j + 4 <= dim; j += 4) {
    float v[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) v[q] = x(j + q);
#pragma unroll
    for (int q = 0; q < 4; ++q)
#pragma unroll
      for (int l = 0; l < kGroup; ++l) {
        const float d = v[q] - row[l][j + q];
        acc[l] = acc[l] + d * d;
      }
  }
  for (; j < dim; ++j) {
    const float v = x(j);
#pragma unroll
    for (int l = 0; l < kGroup; ++l) {
      const float d = v - row[l][j];
      acc[l] = acc[l] + d * d;
    }
  }
}

}  // namespace

template <int TIE>
__global__ void __launch_bounds__(kRoundsThreads) fps_rounds_any(RoundsParams) {
  constexpr int W = kRoundsThreads / 64;
  constexpr int CAP = (int)kAnyCap;
  constexpr int LIST = 2 * CAP;
  constexpr int CH = CAP / 64;
  extern __shared__ float s_any[];  // CAP rows of coordinates, then the min-distances
  __shared__ RoundsCounts S;
  __shared__ alignas(16) uint64_t s_ck[LIST];
  __shared__ uint32_t s_rank[LIST];
  __shared__ uint64_t s_sk[CAP];
  __shared__ uint64_t s_lk[CAP];
  __shared__ uint8_t s_low[CAP / 32][CAP][4];
  __shared__ uint64_t s_acc[CH];
  __shared__ uint32_t s_pp[CAP];  // the picks' rows
  __shared__ uint32_t s_pt[CAP];  // and tie words

  ParamsPtr params = (ParamsPtr)__builtin_amdgcn_kernarg_segment_ptr();  // the only argument
  int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const uint32_t G = gridDim.x;
  const uint32_t g = blockIdx.x;
  const uint32_t nbl = (params->nblocks - g + G - 1) / G;  // blocks g, g + G, ... of 64 points
  const uint32_t dim = params->fps.dim;
  const uint32_t pitch = dim | 1u;  // odd: lanes reading 64 rows meet 64 banks in turn
  float *rows = s_any;
  int *s_dm = (int *)(s_any + (size_t)CAP * pitch);

  if (tid == 0) {
    S.clear(0);
    S.clear(1);
    S.stuck = 0;
    S.ok = 1;
  }
  for (uint32_t q = tid; q < nbl * 64; q += kRoundsThreads)
    s_dm[q] = ((q >> 6) * G + g) * 64 + (q & 63) < params->fps.n
                  ? __float_as_int(params->fps.init)
                  : __float_as_int(-1.0f);

  uint32_t s = 0, np = 0;
  uint64_t T = ~0ull, Tg = ~0ull;
  uint64_t step = (uint64_t)1 << 51;
  uint32_t e = 0, empty = 0;

  // Coordinates of the point with tie word t into row r, by one wave.
  auto fetch = [&](uint32_t r, uint32_t t) {
    const size_t i = tie_of<TIE>(t);
    const __attribute__((address_space(4))) FpsParams &f = params->fps;
    const float *p = f.pts + i * f.sp;
    for (uint32_t j = tid & 63; j < dim; j += 64) rows[r * pitch + j] = p[(size_t)j * f.ld];
  };

  for (;;) {
    asm volatile("" : "+v"(tid), "+s"(params));
    const __attribute__((address_space(4))) RoundsParams &a = *params;
    const __attribute__((address_space(4))) FpsParams &f = a.fps;
    const int lane = tid & 63;
    // The same in every lane (see fps_rounds.hip).
    s = uniform_u32(s);
    np = uniform_u32(np);
    e = uniform_u32(e);
    empty = uniform_u32(empty);
    T = uniform_u64(T);
    Tg = uniform_u64(Tg);
    step = uniform_u64(step);
    // ---- forced picks -------------------------------------------------------
    if (s < f.n_starts) {
      np = min(f.n_starts - s, (uint32_t)CAP);
      for (uint32_t q = tid; q < np; q += kRoundsThreads) {
        uint64_t idx = f.starts[s + q];
        if (idx >= f.n) {
          atomicOr(f.status, kStatusBadStart);
          idx = 0;
        }
        s_pp[q] = q;
        s_pt[q] = tie_of<TIE>((uint32_t)idx);
      }
      __syncthreads();
      for (uint32_t q = wave; q < np; q += W) fetch(q, s_pt[q]);
      __syncthreads();
    }
    // ---- record -------------------------------------------------------------
    if (g == 0) {
      for (uint32_t q = tid; q < np; q += kRoundsThreads) f.out[s + q] = tie_of<TIE>(s_pt[q]);
      if (f.out_pts != nullptr)
        for (uint32_t q = wave; q < np; q += W)
          for (uint32_t j = lane; j < dim; j += 64)
            f.out_pts[(size_t)(s + q) * dim + j] = rows[s_pp[q] * pitch + j];
      if (tid == 0) f.status[1] = e;
    }
    s += np;
    if (s >= f.m) return;
    if (uniform_u32(np && S.stuck)) {
      // The last pick left its own key unchanged, so it stays the best for good.
      if (g == 0) {
        const uint32_t t = s_pt[np - 1], r = s_pp[np - 1];
        for (uint32_t q = s + tid; q < f.m; q += kRoundsThreads) f.out[q] = tie_of<TIE>(t);
        if (f.out_pts != nullptr)
          for (uint32_t q = s + wave; q < f.m; q += W)
            for (uint32_t j = lane; j < dim; j += 64)
              f.out_pts[(size_t)q * dim + j] = rows[r * pitch + j];
      }
      return;
    }
    const bool gather = s >= f.n_starts;
    if (!gather) Tg = ~0ull;

    // ---- update: eight picks on 64 points a job -----------------------------
    const uint32_t groups = (np + kGroup - 1) / kGroup;
    for (uint32_t job = wave; job < nbl * groups; job += W) {
      const uint32_t pg = job / nbl, lb = job - pg * nbl;
      const uint32_t i = (lb * G + g) * 64 + lane;
      const float *p = a.rest + min(i, f.n - 1);
      const float *row[kGroup];
#pragma unroll
      for (int l = 0; l < kGroup; ++l)
        row[l] = rows + (uint32_t)__builtin_amdgcn_readfirstlane(
                            (int)(s_pp[min(pg * kGroup + l, np - 1)] * pitch));
      float acc[kGroup];
      group_dist([&](uint32_t j) { return p[(size_t)j * f.n]; }, row, dim, acc);
      float m = INFINITY;
#pragma unroll
      for (int l = 0; l < kGroup; ++l) m = min_keep(acc[l], m);
      // (both are bit patterns of values from +0 up, which order as integers)
      if (i < f.n) atomicMin(&s_dm[lb * 64 + lane], __float_as_int(m));
    }
    __syncthreads();
    if (!gather) continue;
    uint64_t wmax = 0;
    const int tv = (int)(uint32_t)(Tg >> 32) - 1;
    const uint32_t tt = (uint32_t)Tg;
    for (uint32_t lb = wave; lb < nbl; lb += W) {
      const int b = s_dm[lb * 64 + lane];
      const uint32_t tie = tie_of<TIE>((lb * G + g) * 64 + lane);
      const int wv = wave_max_i32(b);
      const uint64_t bkey = make_key(wv, wave_max_u32(b == wv ? tie : 0u));
      if (bkey > Tg) {
        const bool c = b > tv || (b == tv && tie > tt);
        const uint64_t m = __ballot(c);
        uint32_t at = 0;
        if (lane == 0) at = atomicAdd(&S.cnt[(e + 1) & 1], (uint32_t)__popcll(m));
        at = (uint32_t)__builtin_amdgcn_readfirstlane((int)at) + lanes_below(m);
        if (c && at < (uint32_t)CAP) s_lk[at] = make_key(b, tie);
      }
      wmax = bkey > wmax ? bkey : wmax;
    }
    if (lane == 0) S.wmax[wave] = wmax;
    if (tid < LIST) {
      s_ck[tid] = 0;
      s_rank[tid] = 0;
    }
    lds_barrier();
    ++e;
    const uint32_t par = e & 1u;
    const uint32_t own = S.cnt[par];
    uint64_t U = wave_max_u64(lane < W ? S.wmax[lane] : 0ull);

    // ---- exchange -----------------------------------------------------------
    uint32_t C = own;
    if (G > 1) {
      if (!rounds_exchange<0, LIST>(f.xchg, f.spin_ticks, a.cap_wg, G, g, e, tid, wave, S, s_lk,
                                    (const Rec<0> *)nullptr, s_ck, (Rec<0> *)nullptr, C, U)) {
        if (tid == 0) atomicOr(f.status, kStatusTimeout);
        return;
      }
    } else {
      if ((uint32_t)tid < own && tid < CAP) s_ck[tid] = s_lk[tid];
      if (own > (uint32_t)CAP) C = max(own, (uint32_t)LIST + 1);
      lds_barrier();
    }
    if (tid == 0) S.clear(par ^ 1);  // everybody has read the last round's
    U = uniform_u64(U);
    C = (uint32_t)__builtin_amdgcn_readfirstlane((int)C);
    if (C > (uint32_t)LIST || C == 0) {
      // Too many candidates, or none: the best point of all is the pick (see fps_rounds.hip).
      if (wave == 0) {
        fetch(0, (uint32_t)U);
        bool own = true;  // (a coordinate without a distance to itself leaves the point as it is)
        for (uint32_t j = lane; j < dim; j += 64) own = own && rows[j] - rows[j] == 0.0f;
        if (lane == 0) {
          s_pp[0] = 0;
          s_pt[0] = (uint32_t)U;
        }
        if (__ballot(!own) || !(0.0f < __int_as_float((int)(uint32_t)(U >> 32) - 1)))
          if (lane == 0) S.stuck = 1;
      }
      np = 1;
      if (C)
        step = less_step(step, a.target, C);
      else if (empty)
        step = next_step(step, a.target, 1);
      empty = C == 0;
      T = U;
      Tg = round_bound(T, step);
      __syncthreads();
      continue;
    }

    // ---- front --------------------------------------------------------------
    rank_candidates(s_ck, s_rank, C, tid, wave);
    lds_barrier();
    if ((uint32_t)tid < C) {
      const uint32_t r = s_rank[tid];
      if (r < (uint32_t)CAP)
        s_sk[r] = s_ck[tid];
      else if (r == (uint32_t)CAP)
        S.te[par] = s_ck[tid];  // the first one that the front does not see is the bound
    }
    lds_barrier();
    const uint32_t F = min(C, (uint32_t)CAP);
    const uint32_t nc = (F + 63u) >> 6;
    for (uint32_t r = wave; r < F; r += W)
      fetch(r, (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)s_sk[r]));
    __syncthreads();
    for (uint32_t job = wave, c = 0; c < nc;) {
      if (job >= 8 * (c + 1)) {
        job -= 8 * (c + 1);
        ++c;
        continue;
      }
      const uint32_t j0 = job * kGroup;
      if (j0 < F) {
        const uint32_t i = c * 64 + lane;
        const float v = __int_as_float((int)(uint32_t)(s_sk[i] >> 32) - 1);
        const float *xi = rows + min(i, F - 1) * pitch;
        const float *row[kGroup];
#pragma unroll
        for (int l = 0; l < kGroup; ++l) row[l] = rows + min(j0 + l, F - 1) * pitch;
        float acc[kGroup];
        group_dist([&](uint32_t j) { return xi[j]; }, row, dim, acc);
        uint32_t bits = 0;
#pragma unroll
        for (int l = 0; l < kGroup; ++l) bits |= acc[l] < v ? 1u << l : 0u;
        s_low[job >> 2][i][job & 3] = (uint8_t)bits;
      }
      job += W;
    }
    lds_barrier();
    const uint32_t *low = (const uint32_t *)&s_low[0][0][0];
    if (wave == 0) settle_candidates<CAP>(low, F, lane, s_acc);
    if (wave == 1 && lane == 0) S.step = next_step(step, a.target, C);  // (in its shadow)
    lds_barrier();
    uint64_t key = 0, taken = 0;
    if ((uint32_t)wave < nc) {
      const uint32_t i = (uint32_t)tid;
      key = s_sk[i];
      const float v = __int_as_float((int)(uint32_t)(key >> 32) - 1);
      taken = uniform_u64(s_acc[wave]);
      const bool mine = (taken >> lane) & 1;
      int by = -1;
#pragma unroll
      for (int w = CH - 1; w >= 0; --w) {
        if (w <= wave) {
          uint64_t k = ((uint64_t)low[(2 * w + 1) * CAP + i] << 32) | low[2 * w * CAP + i];
          if (w == wave) k &= ((uint64_t)1 << lane) - 1;
          k &= s_acc[w];
          if (k) by = w * 64 + __ffsll((unsigned long long)k) - 1;
        }
      }
      if (i < F && (mine || by >= 0)) {
        // A candidate partly lowered raises the bound; a pick that does not lower itself
        // ends the round.
        const float *xi = rows + i * pitch, *xb = rows + (mine ? i : (uint32_t)by) * pitch;
        float d = 0.0f;
        for (uint32_t j = 0; j < dim; ++j) {
          const float df = xi[j] - xb[j];
          d = d + df * df;
        }
        if (mine) {
          if (!(d < v)) atomicMin(&S.stop[par], i);
        } else {
          const uint64_t nk = make_key(__float_as_int(d), (uint32_t)key);
          if (nk > Tg) atomicMax((unsigned long long *)&S.te[par], (unsigned long long)nk);
        }
      }
    }
    lds_barrier();
    T = uniform_u64(S.te[par]);
    T = T > Tg ? T : Tg;
    if ((uint32_t)wave < nc) {
      const uint32_t stop = S.stop[par];
      uint32_t at = 0;
      for (int w = 0; w < wave; ++w) at += (uint32_t)__popcll(s_acc[w]);
      taken &= __ballot(key > T && (uint32_t)tid <= stop);
      at = (uint32_t)__builtin_amdgcn_readfirstlane((int)at);
      const uint32_t room = f.m - s;
      if (taken) {
        const uint32_t q = at + lanes_below(taken);
        if (((taken >> lane) & 1) && q < room) {
          s_pt[q] = (uint32_t)key;
          s_pp[q] = (uint32_t)tid;
        }
        if (lane == 0) atomicMax(&S.np[par], min(at + (uint32_t)__popcll(taken), room));
        if (stop - (uint32_t)wave * 64 < 64u && ((taken >> (stop & 63u)) & 1) && lane == 0)
          S.stuck = 1;
      }
    }
    lds_barrier();
    empty = 0;
    np = uniform_u32(S.np[par]);
    step = uniform_u64(S.step);
    Tg = round_bound(T, step);
  }
}

static const KernelEntry kAny[] = {
    {0, kRoundsThreads, 1, kTieHighest, (const void *)fps_rounds_any<kTieHighest>},
    {0, kRoundsThreads, 1, kTieLowest, (const void *)fps_rounds_any<kTieLowest>},
};

const KernelEntry *rounds_any_kernel(int tie) { return &kAny[tie == kTieHighest ? 0 : 1]; }

}  // namespace fpsx
