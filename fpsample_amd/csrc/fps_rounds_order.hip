// fps_rounds_order.hip -- spatial order of a cloud for the threshold rounds.
//
// The rounds only ask that the points of a block lie close together: the picks do not depend
// on the order (ties go by original index), so neither a full sort nor a stable one is
// needed.  The order follows the Hilbert index of the first three coordinates, 10 bits each
// over the bounding box.
//   up to kChunk points: one workgroup does it all in one launch;
//   beyond: the box; a count of every workgroup's points per bucket (the curve's coarse
//   cells); a scan of the counts; the scatter into buckets; and a counting sort of every
//   kChunk consecutive records by as fine a stretch of the curve as their range allows.
// Every step gives each workgroup equally many points, however they cluster.  Only kernels
// are launched (no memset, no copy), so the sequence can be captured.
//
// It writes records {x, y, z, original index} (16 bytes, one load for a point) and, beyond
// three dimensions, the further coordinates as one array each.
#include <hip/hip_runtime.h>

#include "fps_device.hpp"
#include "fps_rounds.hpp"
#include "fpsx.h"
#include "fpsx_curve.hpp"
#include "fpsx_internal.hpp"

#include <algorithm>
#include <string>

namespace fpsx {

struct RoundsOrderScratch {
  DevBuf part, hist, tmp;
};

RoundsOrderScratch *new_rounds_order_scratch() { return new RoundsOrderScratch(); }

void delete_rounds_order_scratch(RoundsOrderScratch *S) {
  if (!S) return;
  for (DevBuf *b : {&S->part, &S->hist, &S->tmp}) b->free();
  delete S;
}

void hold_rounds_order_scratch(RoundsOrderScratch *S) {
  if (!S) return;
  for (DevBuf *b : {&S->part, &S->hist, &S->tmp}) b->held = b->p != nullptr;
}

namespace {

constexpr int kThreads = 1024;
constexpr int kPer = 8;                     // records of a thread in the last step
constexpr uint32_t kChunk = kThreads * kPer;
constexpr uint32_t kBins = 4096;            // counters of the last step
constexpr uint32_t kBoxGroups = 256;
constexpr int kCoarse = 4;                  // bits per axis of the buckets
constexpr uint32_t kMaxBuckets = 1u << (3 * kCoarse);

struct Cloud {
  const float *pts;
  uint64_t sp, ld;
  uint32_t n, dim;
};

// Up to three coordinates of point i (0 beyond the cloud's dimension).
__device__ __forceinline__ void load3(const Cloud &c, uint32_t i, float (&x)[3]) {
#pragma unroll
  for (int j = 0; j < 3; ++j)
    x[j] = (uint32_t)j < c.dim ? c.pts[(size_t)i * c.sp + (size_t)j * c.ld] : 0.0f;
}

// Minimum and maximum of three values over the workgroup, in every thread.
__device__ __forceinline__ void group_box(float (&lo)[3], float (&hi)[3], float (*s)[6]) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
#pragma unroll
  for (int j = 0; j < 3; ++j) {
    lo[j] = wave_min_f(lo[j]);
    hi[j] = wave_max_f(hi[j]);
    if (lane == 0) {
      s[wave][j] = lo[j];
      s[wave][3 + j] = hi[j];
    }
  }
  __syncthreads();
  const int w = lane % (int)(blockDim.x >> 6);
#pragma unroll
  for (int j = 0; j < 3; ++j) {
    lo[j] = wave_min_f(s[w][j]);
    hi[j] = wave_max_f(s[w][3 + j]);
  }
  __syncthreads();
}

// The Hilbert index of a point's cell, of its first BITS bits per axis.
template <int BITS>
__device__ __forceinline__ uint32_t curve_code(const float (&x)[3], const float (&lo)[3],
                                               const float (&hi)[3]) {
  uint32_t q[3];
#pragma unroll
  for (int j = 0; j < 3; ++j) {
    const float span = hi[j] - lo[j];
    const float scale = (span > 0.0f && span < INFINITY) ? 1023.0f / span : 0.0f;
    float v = (x[j] - lo[j]) * scale;
    if (!(v >= 0.0f)) v = 0.0f;  // NaN and anything below the box
    if (v > 1023.0f) v = 1023.0f;
    q[j] = (uint32_t)v >> (10 - BITS);
  }
  return hilbert<BITS>(q[0], q[1], q[2]);
}

// The whole cloud's box from the partial ones, in every thread.
__device__ __forceinline__ void whole_box(const float *part, uint32_t groups, float (&lo)[3],
                                          float (&hi)[3], float (*s)[6]) {
#pragma unroll
  for (int j = 0; j < 3; ++j) {
    lo[j] = INFINITY;
    hi[j] = -INFINITY;
  }
  for (uint32_t b = threadIdx.x; b < groups; b += blockDim.x) {
#pragma unroll
    for (int j = 0; j < 3; ++j) {
      lo[j] = fminf(lo[j], part[b * 6 + j]);
      hi[j] = fmaxf(hi[j], part[b * 6 + 3 + j]);
    }
  }
  group_box(lo, hi, s);
}

__global__ void __launch_bounds__(kThreads) order_box(Cloud c, float *part) {
  __shared__ float s[kThreads / 64][6];
  float lo[3] = {INFINITY, INFINITY, INFINITY}, hi[3] = {-INFINITY, -INFINITY, -INFINITY};
  for (uint64_t i = (uint64_t)blockIdx.x * kThreads + threadIdx.x; i < c.n;
       i += (uint64_t)gridDim.x * kThreads) {
    float x[3];
    load3(c, (uint32_t)i, x);
#pragma unroll
    for (int j = 0; j < 3; ++j) {
      lo[j] = fminf(lo[j], x[j]);
      hi[j] = fmaxf(hi[j], x[j]);
    }
  }
  group_box(lo, hi, s);
  if (threadIdx.x == 0) {
#pragma unroll
    for (int j = 0; j < 3; ++j) {
      part[blockIdx.x * 6 + j] = lo[j];
      part[blockIdx.x * 6 + 3 + j] = hi[j];
    }
  }
}

// Points of workgroup g: [g * per, min(n, (g + 1) * per)).  hist[b * G + g]: its count in
// bucket b, so that the scan over hist gives every workgroup its place in every bucket.
__global__ void __launch_bounds__(kThreads)
    order_count(Cloud c, const float *part, uint32_t groups, uint32_t per, int shift,
                uint32_t buckets, uint32_t *hist) {
  __shared__ float s[kThreads / 64][6];
  __shared__ uint32_t s_n[kMaxBuckets];
  float lo[3], hi[3];
  whole_box(part, groups, lo, hi, s);
  for (uint32_t b = threadIdx.x; b < buckets; b += kThreads) s_n[b] = 0;
  __syncthreads();
  const uint64_t end = min((uint64_t)c.n, ((uint64_t)blockIdx.x + 1) * per);
  for (uint64_t i = (uint64_t)blockIdx.x * per + threadIdx.x; i < end; i += kThreads) {
    float x[3];
    load3(c, (uint32_t)i, x);
    atomicAdd(&s_n[curve_code<kCoarse>(x, lo, hi) >> shift], 1u);
  }
  __syncthreads();
  for (uint32_t b = threadIdx.x; b < buckets; b += kThreads)
    hist[(size_t)b * gridDim.x + blockIdx.x] = s_n[b];
}

// Exclusive prefix sum over the workgroup's values, one per thread.
__device__ __forceinline__ uint32_t group_scan(uint32_t v, uint32_t *s) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const uint32_t x = wave_scan_add(v);
  if (lane == 63) s[wave] = x;
  __syncthreads();
  uint32_t before = 0;
  for (int w = 0; w < wave; ++w) before += s[w];
  return before + x - v;
}

// In-place exclusive scan of each bucket's counts over the workgroups (one wave a bucket, at
// most 256 counts) and the bucket's total.
__global__ void __launch_bounds__(kThreads)
    order_scan(uint32_t *hist, uint32_t g, uint32_t buckets, uint32_t *total) {
  const uint32_t lane = threadIdx.x & 63;
  const uint32_t b = blockIdx.x * (kThreads / 64) + (threadIdx.x >> 6);
  if (b >= buckets) return;
  uint32_t *h = hist + (size_t)b * g;
  uint32_t v[4], sum = 0;
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    v[k] = lane * 4 + k < g ? h[lane * 4 + k] : 0u;
    sum += v[k];
  }
  const uint32_t incl = wave_scan_add(sum);
  uint32_t x = incl - sum;
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    if (lane * 4 + k < g) h[lane * 4 + k] = x;
    x += v[k];
  }
  if (lane == 63) total[b] = incl;
}

__global__ void __launch_bounds__(kThreads)
    order_scatter(Cloud c, const float *part, uint32_t groups, uint32_t per, int shift,
                  uint32_t buckets, const uint32_t *hist, const uint32_t *total, float4 *rec) {
  __shared__ float s[kThreads / 64][6];
  __shared__ uint32_t s_sum[kThreads / 64];
  __shared__ uint32_t s_at[kMaxBuckets];
  float lo[3], hi[3];
  whole_box(part, groups, lo, hi, s);
  constexpr int K = kMaxBuckets / kThreads;
  uint32_t v[K], sum = 0;
#pragma unroll
  for (int k = 0; k < K; ++k) {
    const uint32_t b = threadIdx.x * K + k;
    v[k] = b < buckets ? total[b] : 0u;
    sum += v[k];
  }
  uint32_t x0 = group_scan(sum, s_sum);
#pragma unroll
  for (int k = 0; k < K; ++k) {
    const uint32_t b = threadIdx.x * K + k;
    if (b < buckets) s_at[b] = x0 + hist[(size_t)b * gridDim.x + blockIdx.x];
    x0 += v[k];
  }
  __syncthreads();
  const uint64_t end = min((uint64_t)c.n, ((uint64_t)blockIdx.x + 1) * per);
  for (uint64_t i = (uint64_t)blockIdx.x * per + threadIdx.x; i < end; i += kThreads) {
    float x[3];
    load3(c, (uint32_t)i, x);
    const uint32_t at = atomicAdd(&s_at[curve_code<kCoarse>(x, lo, hi) >> shift], 1u);
    rec[at] = make_float4(x[0], x[1], x[2], __int_as_float((int)i));
  }
}

// Counting sort of the kChunk records from base on (in: already in buckets; null: the cloud
// itself, in the box of these points) along the curve.
__device__ __forceinline__ void chunk_order(const Cloud &c, const uint32_t base, const float *part,
                                            uint32_t groups, const float4 *in, float4 *out,
                                            float *rest) {
  __shared__ float s[kThreads / 64][6];
  __shared__ uint32_t s_sum[kThreads / 64];
  __shared__ uint32_t s_n[kBins];
  __shared__ uint32_t s_lo, s_hi;
  const uint32_t count = min(kChunk, c.n - base);
  float4 r[kPer];
#pragma unroll
  for (int k = 0; k < kPer; ++k) {
    const uint32_t q = min((uint32_t)(k * kThreads + threadIdx.x), count - 1);
    if (in) {
      r[k] = in[base + q];
    } else {
      float x[3];
      load3(c, base + q, x);
      r[k] = make_float4(x[0], x[1], x[2], __int_as_float((int)(base + q)));
    }
  }
  float lo[3], hi[3];
  if (in) {
    whole_box(part, groups, lo, hi, s);
  } else {
#pragma unroll
    for (int j = 0; j < 3; ++j) {
      lo[j] = INFINITY;
      hi[j] = -INFINITY;
    }
#pragma unroll
    for (int k = 0; k < kPer; ++k) {
      const float x[3] = {r[k].x, r[k].y, r[k].z};
#pragma unroll
      for (int j = 0; j < 3; ++j) {
        lo[j] = fminf(lo[j], x[j]);
        hi[j] = fmaxf(hi[j], x[j]);
      }
    }
    group_box(lo, hi, s);
  }
  uint32_t code[kPer], cl = ~0u, ch = 0;
#pragma unroll
  for (int k = 0; k < kPer; ++k) {
    const float x[3] = {r[k].x, r[k].y, r[k].z};
    code[k] = curve_code<10>(x, lo, hi);
    cl = min(cl, code[k]);
    ch = max(ch, code[k]);
  }
  if (threadIdx.x == 0) {
    s_lo = ~0u;
    s_hi = 0;
  }
  for (uint32_t b = threadIdx.x; b < kBins; b += kThreads) s_n[b] = 0;
  __syncthreads();
  cl = ~wave_max_u32(~cl);
  ch = wave_max_u32(ch);
  if ((threadIdx.x & 63) == 0) {
    atomicMin(&s_lo, cl);
    atomicMax(&s_hi, ch);
  }
  __syncthreads();
  cl = s_lo;
  int shift = 0;
  while (((s_hi - cl) >> shift) >= kBins) ++shift;
  uint32_t rank[kPer];
#pragma unroll
  for (int k = 0; k < kPer; ++k) {
    code[k] = (code[k] - cl) >> shift;
    rank[k] = (uint32_t)(k * kThreads + threadIdx.x) < count ? atomicAdd(&s_n[code[k]], 1u) : 0u;
  }
  __syncthreads();
  uint32_t v[kBins / kThreads], sum = 0;
#pragma unroll
  for (int k = 0; k < (int)(kBins / kThreads); ++k) {
    v[k] = s_n[threadIdx.x * (kBins / kThreads) + k];
    sum += v[k];
  }
  uint32_t at = group_scan(sum, s_sum);
#pragma unroll
  for (int k = 0; k < (int)(kBins / kThreads); ++k) {
    s_n[threadIdx.x * (kBins / kThreads) + k] = at;
    at += v[k];
  }
  __syncthreads();
#pragma unroll
  for (int k = 0; k < kPer; ++k) {
    if ((uint32_t)(k * kThreads + threadIdx.x) >= count) continue;
    const uint32_t p = base + s_n[code[k]] + rank[k];
    out[p] = r[k];
    const uint32_t i = (uint32_t)__float_as_int(r[k].w);
    for (uint32_t j = 3; j < c.dim; ++j)
      rest[(size_t)(j - 3) * c.n + p] = c.pts[(size_t)i * c.sp + (size_t)j * c.ld];
  }
}

__global__ void __launch_bounds__(kThreads)
    order_chunk(Cloud c, const float *part, uint32_t groups, const float4 *in, float4 *out,
                float *rest) {
  chunk_order(c, blockIdx.x * kChunk, part, groups, in, out, rest);
}

__global__ void __launch_bounds__(kThreads) order_pieces(const RoundsOrderJob *jobs) {
  const RoundsOrderJob j = jobs[blockIdx.x];
  const Cloud c = {j.pts, j.sp, j.ld, j.n, j.dim};
  chunk_order(c, j.base, nullptr, 0, nullptr, j.rec, j.rest);
}

}  // namespace

#define HIP_OR_FAIL(expr)                                              \
  do {                                                                 \
    hipError_t _e = (expr);                                            \
    if (_e != hipSuccess)                                              \
      return fail(_e == hipErrorOutOfMemory ? FPSX_ENOMEM : FPSX_EHIP, \
                  std::string(#expr) + ": " + hipGetErrorString(_e));  \
  } while (0)

namespace {

// Buckets of about 2048 points, at most kMaxBuckets; count and scatter by at most 256
// workgroups of 4096 points and more.
int bucket_bits(uint32_t n) {
  int bits = 5;
  while (bits < 3 * kCoarse && (n >> (bits + 11)) != 0) ++bits;
  return bits;
}
uint32_t count_groups(uint32_t n) { return std::min<uint32_t>(256, (n + 4095) / 4096); }

}  // namespace

int rounds_order_reserve(RoundsOrderScratch &S, uint32_t n) {
  if (n <= kChunk) return FPSX_OK;
  const size_t buckets = (size_t)1 << bucket_bits(n);
  HIP_OR_FAIL(S.part.reserve(kBoxGroups * 6 * sizeof(float)));
  HIP_OR_FAIL(S.hist.reserve(buckets * (count_groups(n) + 1) * sizeof(uint32_t)));
  HIP_OR_FAIL(S.tmp.reserve((size_t)n * sizeof(float4)));
  return FPSX_OK;
}

bool rounds_order_ready(const RoundsOrderScratch *S, uint32_t n) {
  if (n <= kChunk) return true;
  const size_t buckets = (size_t)1 << bucket_bits(n);
  return S && S->part.cap >= kBoxGroups * 6 * sizeof(float) &&
         S->hist.cap >= buckets * (count_groups(n) + 1) * sizeof(uint32_t) &&
         S->tmp.cap >= (size_t)n * sizeof(float4);
}

int rounds_order(const float *pts, uint64_t sp, uint64_t ld, uint32_t n, uint32_t dim, float4 *rec,
                 float *rest, RoundsOrderScratch &S, hipStream_t st) {
  const Cloud c = {pts, sp, ld, n, dim};
  const uint32_t chunks = (n + kChunk - 1) / kChunk;
  if (chunks == 1) {
    hipLaunchKernelGGL(order_chunk, dim3(1), dim3(kThreads), 0, st, c, nullptr, 0u, nullptr, rec,
                       rest);
    HIP_OR_FAIL(hipGetLastError());
    return FPSX_OK;
  }
  const int bits = bucket_bits(n);
  const uint32_t buckets = 1u << bits;
  const uint32_t g = count_groups(n);
  const uint32_t per = (n + g - 1) / g;
  const uint32_t gb = std::min<uint32_t>(kBoxGroups, (n + 2047) / 2048);
  const int rc = rounds_order_reserve(S, n);
  if (rc) return rc;
  float *part = (float *)S.part.p;
  uint32_t *hist = (uint32_t *)S.hist.p, *total = hist + (size_t)buckets * g;
  const int shift = 3 * kCoarse - bits;
  hipLaunchKernelGGL(order_box, dim3(gb), dim3(kThreads), 0, st, c, part);
  HIP_OR_FAIL(hipGetLastError());
  hipLaunchKernelGGL(order_count, dim3(g), dim3(kThreads), 0, st, c, part, gb, per, shift,
                     buckets, hist);
  HIP_OR_FAIL(hipGetLastError());
  hipLaunchKernelGGL(order_scan, dim3((buckets + kThreads / 64 - 1) / (kThreads / 64)),
                     dim3(kThreads), 0, st, hist, g, buckets, total);
  HIP_OR_FAIL(hipGetLastError());
  hipLaunchKernelGGL(order_scatter, dim3(g), dim3(kThreads), 0, st, c, part, gb, per, shift,
                     buckets, hist, total, (float4 *)S.tmp.p);
  HIP_OR_FAIL(hipGetLastError());
  hipLaunchKernelGGL(order_chunk, dim3(chunks), dim3(kThreads), 0, st, c, part, gb,
                     (const float4 *)S.tmp.p, rec, rest);
  HIP_OR_FAIL(hipGetLastError());
  return FPSX_OK;
}

void rounds_order_pieces(const float *pts, uint64_t sp, uint64_t ld, uint32_t n, uint32_t dim,
                         float4 *rec, float *rest, std::vector<RoundsOrderJob> &jobs) {
  for (uint64_t base = 0; base < n; base += kChunk)
    jobs.push_back({pts, sp, ld, rec, rest, n, dim, (uint32_t)base});
}

hipError_t launch_order_pieces(const RoundsOrderJob *jobs, uint32_t count, hipStream_t st) {
  hipLaunchKernelGGL(order_pieces, dim3(count), dim3(kThreads), 0, st, jobs);
  return hipGetLastError();
}

}  // namespace fpsx
