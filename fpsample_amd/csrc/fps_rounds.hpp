// fps_rounds.hpp -- host-visible description of the threshold-round FPS kernel.
#pragma once
#include <hip/hip_runtime.h>
#include <stddef.h>
#include <stdint.h>

#include <vector>

#include "fps_kernels.hpp"

namespace fpsx {

struct RoundsParams {
  FpsParams fps;       // the cloud (original order), picks, exchange area, status, dmin
  // The points in spatial order: {x, y, z, original index} of every position, and coordinate
  // j >= 3 at rest[(j - 3) * n + position].  Null: positions are indices, points as in fps.
  const float4 *rec;
  const float *rest;
  uint32_t nblocks;      // blocks of 64 * P consecutive positions
  uint32_t cap_wg;       // candidates one workgroup may publish per round
  uint32_t target;       // candidates aimed at per round
  // Picks s_begin .. s_end - 1 of fps.m.  s_begin > 0 continues a run whose min-distances
  // fps.dmin holds by position, with every pick so far applied; s_end < fps.m saves them so.
  uint32_t s_begin, s_end;
  uint32_t *carry;       // four words kept from one part of such a run to the next
  uint64_t start;        // pick 0 where fps.starts is null
  // One cloud of several (fps_rounds_jobs): its workgroups, the first one's slot, and a
  // counter of those that have claimed it, zeroed before the launch.
  uint32_t team, member_base;
  uint32_t *ready;
  uint64_t form_ticks;    // bound on the wait of the first exchange
  uint32_t *host_status;  // where not null, a host word that a failure is stored to as well
};

// Any dimension (fps_rounds_any.hip): candidates a round decides on; rest holds the points by
// coordinate (j at rest[j * n + i]), rec is unused.
constexpr uint32_t kAnyCap = 128;
constexpr uint32_t kAnyMaxDim = 256;
inline size_t rounds_any_shmem(uint32_t dim, uint32_t nbl) {
  return ((size_t)kAnyCap * (dim | 1u) + (size_t)nbl * 64) * sizeof(float);
}
const KernelEntry *rounds_any_kernel(int tie);

struct RoundsJobs {
  const RoundsParams *table;
  const uint32_t *member_job;  // slot -> entry of table
  uint32_t members;
  uint32_t *claim;             // zeroed before the launch
  uint64_t team_ticks;         // bound on a team's forming
  uint32_t one_slot;           // one workgroup per slot, all co-resident
};

constexpr int kRoundsThreads = 1024;
constexpr uint32_t kRoundsCap = 256;       // candidates a round decides on
constexpr uint32_t kRoundsList = 512;      // candidates that may come in: the best kRoundsCap count
constexpr uint32_t kRoundsMaxGrid = 256;
constexpr uint32_t kRoundsHeadWords = 3;   // count, high and low half of the best key
constexpr uint32_t kRoundsReplicas = 4;    // copies of the headers
// Candidates a round aims at for m picks (fpsx_api.hip has the figures).
inline uint32_t rounds_target(size_t m) {
  return m >= 16384 ? 224 : m >= 1280 ? 160 : m <= 512 ? 64 : (uint32_t)(m / 8);
}
// Candidates one workgroup may publish: a round in which one has more takes one pick, as clustered
// clouds do with small limits, and larger areas cost their clearing and the candidates' way (us a
// run and rounds at 64 / 32 for up to 64 and more workgroups, at 128 / 64 and at 256 / 128: 2^24
// lattice points, 2048 picks 3608 (220), 3321 (168), 3305 (147); 2^20 clustered points, 16384
// picks 2035 (196), 1989 (181), 2027 (171); 2^22 / 4096 1999, 1983, 2040).
inline uint32_t rounds_cap_wg(uint32_t grid) {
  return grid <= 8 ? kRoundsCap : grid <= 64 ? 128 : 64;
}
// Words between the arrays of a header's words: 2 KiB apart they lie on different memory
// channels, which all workgroups' polls then share (64 workgroups, 50 K points: 9.1 us a round
// against 9.6 with the arrays end to end).  Small teams, of which a launch has many, stay close.
constexpr __host__ __device__ uint32_t rounds_head_pitch(uint32_t grid) {
  return grid < 16 ? 16 : 256;
}
// Exchange words of a grid: two buffers of headers and candidates.
inline size_t rounds_xchg_words(uint32_t grid, uint32_t dim, uint32_t cap_wg) {
  if (grid <= 1) return 1;
  return (size_t)2 * ((size_t)kRoundsReplicas * kRoundsHeadWords * rounds_head_pitch(grid) +
                      (size_t)(2 + dim) * grid * cap_wg);
}
// The largest single-cloud area: reserved at once, so that it never moves under a captured call.
inline size_t rounds_xchg_most() {
  const size_t a = rounds_xchg_words(kRoundsMaxGrid, 8, rounds_cap_wg(kRoundsMaxGrid));
  const size_t b = rounds_xchg_words(64, 8, rounds_cap_wg(64));
  return a > b ? a : b;
}
// Dynamic LDS of a workgroup holding nbl blocks: box and best key of each.
inline size_t rounds_shmem(uint32_t dim, uint32_t nbl) {
  return (size_t)nbl * (2 * dim * sizeof(float) + sizeof(uint64_t));
}

const KernelEntry *rounds_table(size_t *count);
// The kernel for many clouds of a dimension (highest-index ties); null beyond four, where a
// batch takes one launch per cloud.
const KernelEntry *rounds_jobs_kernel(int dim);

// Enqueues the spatial order of a cloud (fps_rounds_order.hip): rec holds n records, rest
// (dim - 3) * n floats beyond three dimensions.  Returns a FPSX_* code.
struct RoundsOrderScratch;
RoundsOrderScratch *new_rounds_order_scratch();
void delete_rounds_order_scratch(RoundsOrderScratch *s);
void hold_rounds_order_scratch(RoundsOrderScratch *s);
// Sizes the scratch for clouds of up to n points, so that later calls allocate nothing.
int rounds_order_reserve(RoundsOrderScratch &scratch, uint32_t n);
// Whether a call for n points would allocate nothing.
bool rounds_order_ready(const RoundsOrderScratch *scratch, uint32_t n);
int rounds_order(const float *pts, uint64_t sp, uint64_t ld, uint32_t n, uint32_t dim, float4 *rec,
                 float *rest, RoundsOrderScratch &scratch, hipStream_t st);
// Many clouds in one launch and without scratch: every 8192 consecutive points of a cloud, one
// job of a device table, are ordered among themselves.
struct RoundsOrderJob {
  const float *pts;
  uint64_t sp, ld;
  float4 *rec;
  float *rest;
  uint32_t n, dim, base;
};
void rounds_order_pieces(const float *pts, uint64_t sp, uint64_t ld, uint32_t n, uint32_t dim,
                         float4 *rec, float *rest, std::vector<RoundsOrderJob> &jobs);
hipError_t launch_order_pieces(const RoundsOrderJob *jobs, uint32_t count, hipStream_t st);

}  // namespace fpsx
