// fpsx_batch_internal.hpp -- job tables shared by the batch object and the
// serving loop.
#pragma once
#include <stdint.h>

#include <vector>

#include "fps_batch.hpp"
#include "fps_rounds.hpp"
#include "fpsx_internal.hpp"

namespace fpsx {

// One cloud's work for a launch, before team sizes are chosen.
struct JobSpec {
  uint64_t pt_off, ld, out_off, state_off, start;
  uint32_t n, m, s_begin, s_end;
  uint64_t sorted_off = 0, perm_off = 0;  // pruned kernel: the spatial order
  uint64_t sp = 1;                        // threshold rounds: floats from point to point
};

// Team sizes (ceil(n / min(B * PPT, share_cap))), claim order (teams first,
// longest first) and exchange-area numbering for one launch.  aligned: every
// member's share is exactly B * PPT (the last one takes the rest), as the
// pruned kernel's wave blocks need.
int build_jobs(const JobSpec *specs, size_t n_specs, const KernelEntry *k, uint32_t share_cap,
               std::vector<BatchJob> &jobs, std::vector<uint32_t> &member_job, uint32_t *n_areas,
               bool aligned = false);

// Device tables and scratch of one batch launch.
struct BatchRun {
  const KernelEntry *k = nullptr;
  std::vector<BatchJob> jobs;
  std::vector<uint32_t> member_job;
  uint32_t members = 0;
  uint32_t grid = 0;
  size_t counter_words = 0, xchg_words = 0;
  DevBuf d_jobs, d_member_job, d_counters, d_xchg, d_status;
  BatchParams params;
  // Pruned kernel (fps_batch_pp): its parameters wrap params; one_slot: one
  // workgroup per member slot (grid = members, which must all be co-resident).
  bool pruned = false, one_slot = false;
  BatchPPParams pp_params;
  // Upload tables for this job list (host-synchronous) and fill params.
  // For a pruned kernel, sorted / perm are the bases of BatchJob::sorted_off
  // and ::perm_off.
  int prepare(Ctx &c, const KernelEntry *kernel, const std::vector<BatchJob> &js,
              const std::vector<uint32_t> &mj, uint32_t n_areas, const float *d_pts,
              uint64_t *d_out, float *d_state, const float *sorted = nullptr,
              const uint32_t *perm = nullptr, bool one_slot = false);
  // Clear counters / exchange areas / status and launch (graph-capturable).
  int enqueue(hipStream_t st);
  ~BatchRun() {
    d_jobs.free();
    d_member_job.free();
    d_counters.free();
    d_xchg.free();
    d_status.free();
  }
};

// Where the threshold rounds find a batch's data; a job's offsets (JobSpec) count from these
// bases, sorted_off in floats to the cloud's records and state_off in floats to its
// min-distances by position and four words carried between parts of a run.
struct RoundsBases {
  const float *pts;     // SoA points
  uint64_t *out;
  float *state;
  const float *sorted;  // records {x, y, z, original index}
  const float *rest;    // beyond three dimensions: the further coordinates, at JobSpec::perm_off
};

// The same for the threshold rounds (fps_rounds_jobs).
struct RoundsRun {
  const KernelEntry *k = nullptr;
  uint32_t members = 0, grid = 0;
  size_t shmem = 0, clear_words = 0;
  DevBuf d_tables, d_clear;  // job table and slots; status, claim and team counters, exchange
  RoundsJobs jobs;
  // The tables as built.  one_slot: pinned, with a status word before them that the kernel sets,
  // and copied by the launch itself; no call waits for a copy in either direction.
  std::vector<char> host;
  char *pinned = nullptr;
  size_t pinned_cap = 0, table_words = 0;
  static constexpr size_t kPinnedHead = 64;
  uint32_t host_status() const { return *(volatile uint32_t *)pinned; }
  uint32_t *status() const { return (uint32_t *)d_clear.p; }
  // Tables for these clouds (uploaded host-synchronously unless one_slot).  one_slot: every
  // member has a workgroup of its own, all co-resident, and base_team[i] is the least team of
  // cloud i; the run's last launch has ended.
  int prepare(Ctx &c, int dim, const std::vector<JobSpec> &specs, const RoundsBases &b,
              const std::vector<uint32_t> *base_team = nullptr);
  // (graph-capturable without events, which time the kernel alone and mark its end)
  int enqueue(hipStream_t st, hipEvent_t begin = nullptr, hipEvent_t end = nullptr);
  ~RoundsRun() {
    d_tables.free();
    d_clear.free();
    if (pinned) (void)hipHostFree(pinned);
  }
};

}  // namespace fpsx
