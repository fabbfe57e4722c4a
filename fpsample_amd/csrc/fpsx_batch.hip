// fpsx_batch.hip -- host side of batched FPS: job tables, the batch object
// (device tables + a captured HIP graph of its launch sequence) and its C ABI.
#include <hip/hip_runtime.h>

#include <hip/hip_ext.h>

#include <algorithm>
#include <cfloat>
#include <cmath>
#include <cstdlib>
#include <cstring>
#include <memory>
#include <numeric>
#include <string>
#include <vector>

#include "fps_batch.hpp"
#include "fps_device.hpp"
#include "fpsx.h"
#include "fpsx_batch_internal.hpp"
#include "fpsx_internal.hpp"
#include "fps_pruned.hpp"

#define FPSX_EXPORT extern "C" __attribute__((visibility("default")))

namespace fpsx {

static int hip_err(hipError_t e, const char *what) {
  return fail(e == hipErrorOutOfMemory ? FPSX_ENOMEM : FPSX_EHIP,
              std::string(what) + ": " + hipGetErrorString(e));
}
#define HIP_TRY(expr)                                 \
  do {                                                \
    hipError_t _e = (expr);                           \
    if (_e != hipSuccess) return hip_err(_e, #expr);  \
  } while (0)

static const KernelEntry *find_batch(int dim, int B, int ppt) {
  size_t cnt;
  const KernelEntry *t = batch_table(&cnt);
  for (size_t i = 0; i < cnt; ++i)
    if (t[i].dim == dim && t[i].block == B && t[i].ppt == ppt) return &t[i];
  return nullptr;
}

int build_jobs(const JobSpec *specs, size_t n_specs, const KernelEntry *k, uint32_t share_cap,
               std::vector<BatchJob> &jobs, std::vector<uint32_t> &member_job,
               uint32_t *n_areas, bool aligned) {
  const uint32_t cap = std::min<uint32_t>((uint32_t)(k->block * k->ppt), share_cap ? share_cap : ~0u);
  std::vector<BatchJob> js(n_specs);
  for (size_t c = 0; c < n_specs; ++c) {
    const JobSpec &sp = specs[c];
    BatchJob &J = js[c];
    std::memset(&J, 0, sizeof(J));
    J.pt_off = sp.pt_off;
    J.ld = sp.ld;
    J.out_off = sp.out_off;
    J.state_off = sp.state_off;
    J.start = sp.start;
    J.n = sp.n;
    J.m = sp.m;
    J.s_begin = sp.s_begin;
    J.s_end = sp.s_end;
    J.sorted_off = sp.sorted_off;
    J.perm_off = sp.perm_off;
    uint32_t team = (sp.n + cap - 1) / cap;
    if (team < 1) team = 1;
    if (team > kMaxTeam || team > (uint32_t)k->block)
      return fail(FPSX_ETOOBIG, "cloud of " + std::to_string(sp.n) +
                                    " points exceeds the batch kernel's team capacity");
    J.share = aligned ? cap : (sp.n + team - 1) / team;
    J.team = (sp.n + J.share - 1) / J.share;  // no empty member
  }
  // Teams first (they form at once while the grid is free), then single
  // workgroup jobs; longest first within each group.
  std::vector<size_t> order(n_specs);
  std::iota(order.begin(), order.end(), 0);
  std::stable_sort(order.begin(), order.end(), [&](size_t a, size_t b) {
    const bool ta = js[a].team > 1, tb = js[b].team > 1;
    if (ta != tb) return ta;
    const double wa = (double)js[a].share * (double)(js[a].s_end - js[a].s_begin);
    const double wb = (double)js[b].share * (double)(js[b].s_end - js[b].s_begin);
    return wa > wb;
  });
  jobs.clear();
  member_job.clear();
  uint32_t areas = 0;
  for (size_t o = 0; o < n_specs; ++o) {
    BatchJob J = js[order[o]];
    J.member_base = (uint32_t)member_job.size();
    J.area = (J.team > 1) ? areas++ : 0;
    for (uint32_t r = 0; r < J.team; ++r) member_job.push_back((uint32_t)jobs.size());
    jobs.push_back(J);
  }
  *n_areas = areas;
  return FPSX_OK;
}

int BatchRun::prepare(Ctx &c, const KernelEntry *kernel, const std::vector<BatchJob> &js,
                      const std::vector<uint32_t> &mj, uint32_t n_areas, const float *d_pts,
                      uint64_t *d_out, float *d_state, const float *sorted,
                      const uint32_t *perm, bool one) {
  k = kernel;
  jobs = js;
  member_job = mj;
  members = (uint32_t)mj.size();
  pruned = sorted != nullptr;
  one_slot = one;
  int gmax = c.max_blocks(k, 0);
  if (gmax <= 0) return fail(FPSX_EHIP, "batch kernel cannot be resident");
  if (one_slot && members > (uint32_t)gmax)
    return fail(FPSX_ETOOBIG, "one-slot batch launch: more members than co-resident workgroups");
  grid = std::min<uint32_t>(members, (uint32_t)gmax);
  uint32_t max_team = 1;
  for (auto &J : jobs) max_team = std::max(max_team, J.team);
  if (max_team > grid) return fail(FPSX_ETOOBIG, "a team is larger than the co-resident grid");
  HIP_TRY(d_jobs.reserve(jobs.size() * sizeof(BatchJob)));
  HIP_TRY(d_member_job.reserve(members * sizeof(uint32_t)));
  counter_words = (1 + jobs.size() + 1) / 2 + 1;  // claim + per-job ready counters, in u64 words
  HIP_TRY(d_counters.reserve(counter_words * sizeof(uint64_t)));
  xchg_words = std::max<size_t>(1, (size_t)n_areas * (pruned ? kPPTeamWords : kTeamXchgWords));
  HIP_TRY(d_xchg.reserve(xchg_words * sizeof(uint64_t)));
  HIP_TRY(d_status.reserve(sizeof(uint64_t)));
  HIP_TRY(hipMemcpy(d_jobs.p, jobs.data(), jobs.size() * sizeof(BatchJob),
                    hipMemcpyHostToDevice));
  HIP_TRY(hipMemcpy(d_member_job.p, member_job.data(), members * sizeof(uint32_t),
                    hipMemcpyHostToDevice));
  std::memset(&params, 0, sizeof(params));
  params.pts = d_pts;
  params.jobs = (const BatchJob *)d_jobs.p;
  params.member_job = (const uint32_t *)d_member_job.p;
  params.total_members = members;
  params.claim = (uint32_t *)d_counters.p;
  params.ready = (uint32_t *)d_counters.p + 2;
  params.out = d_out;
  params.state = d_state;
  params.xchg = (uint64_t *)d_xchg.p;
  params.status = (uint32_t *)d_status.p;
  params.init = INFINITY;
  params.spin_ticks = c.spin_ticks;
  params.team_ticks = c.spin_ticks * 5;
  // Teams settle up to two picks per exchange unless FPSX_BATCH_NO_PAIR=1
  // (the one-pick team loop; same picks).
  const char *np = std::getenv("FPSX_BATCH_NO_PAIR");
  params.pair = (np && np[0] == '1') ? 0u : 1u;
  pp_params.b = params;
  pp_params.sorted = sorted;
  pp_params.perm = perm;
  return FPSX_OK;
}

int BatchRun::enqueue(hipStream_t st) {
  HIP_TRY(launch_fill_u64((uint64_t *)d_counters.p, counter_words, 0, st));
  HIP_TRY(launch_fill_u64((uint64_t *)d_xchg.p, xchg_words, 0, st));
  HIP_TRY(launch_fill_u64((uint64_t *)d_status.p, 1, 0, st));
  void *args[] = {pruned ? (void *)&pp_params : (void *)&params};
  HIP_TRY(hipLaunchKernel(k->fn, dim3(grid), dim3(k->block), args, 0, st));
  return FPSX_OK;
}

// Estimated us of one cloud on `team` workgroups: a round costs its front, an exchange beyond
// one workgroup, and 3.6 us for each block of 256 points that a wave updates.  Fitted to us a
// round measured at 1, 2, 4, 8, 16 and 32 workgroups: 65536 points 67, 41, 26, 19, 12 and 11;
// 131072 points 114, 67, 39, 25, 17 and 12; 16384 points 21, 20, 13, 11, 10 and 10.
static double rounds_us(const JobSpec &s, uint32_t target, uint32_t team) {
  const double picks = (double)(s.s_end - s.s_begin);
  const double rounds = 10.0 + picks / (0.55 * target);
  const double share = (double)s.n / (64.0 * 4.0 * 16.0 * team);  // blocks per wave
  return rounds * (7.0 + (team > 1 ? 3.0 : 0.0) + 3.6 * (share > 0.25 ? share : 0.25));
}

// The team sizes to choose from for one cloud: powers of two times the least, while each is
// faster than the ones before, with their times.
struct RoundsTeams {
  uint32_t n = 0;
  uint32_t team[9];
  double us[9];
  uint32_t smallest(double x) const {  // the first that ends within x us, or the fastest
    uint32_t i = 0;
    while (i + 1 < n && us[i] > x) ++i;
    return i;
  }
};

static RoundsTeams rounds_teams(const JobSpec &s, uint32_t target, uint32_t least, uint32_t most) {
  RoundsTeams r;
  for (uint32_t t = least; r.n < 9 && (r.n == 0 || t <= most); t *= 2) {
    const double u = rounds_us(s, target, t);
    if (r.n && u >= r.us[r.n - 1]) continue;
    r.team[r.n] = t;
    r.us[r.n++] = u;
  }
  return r;
}

// The tables of a launch out of host memory, and the clearing of what it counts in.
__global__ void stage_jobs(const uint64_t *tables, uint64_t *dst, size_t words, uint64_t *clear,
                           size_t clear_words) {
  const size_t step = (size_t)gridDim.x * blockDim.x;
  const size_t i0 = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  for (size_t i = i0; i < words; i += step) dst[i] = tables[i];
  for (size_t i = i0; i < clear_words; i += step) clear[i] = 0;
}

int RoundsRun::prepare(Ctx &c, int dim, const std::vector<JobSpec> &specs, const RoundsBases &b,
                       const std::vector<uint32_t> *base_team) {
  const bool one_slot = base_team != nullptr;
  k = rounds_jobs_kernel(dim);
  if (!k) return fail(FPSX_EINVAL, "no threshold-round kernel for this dimension");
  const uint32_t P = (uint32_t)k->ppt;
  const size_t n = specs.size();
  const uint32_t gmax = (uint32_t)c.max_blocks(k, 0);
  std::vector<uint32_t> team(n, 1), target(n), blocks(n);
  std::vector<size_t> order(n);
  std::iota(order.begin(), order.end(), 0);
  for (size_t i = 0; i < n; ++i) {
    const JobSpec &s = specs[i];
    target[i] = rounds_target(s.m);
    blocks[i] = (s.n + 64 * P - 1) / (64 * P);
    // At most 1024 blocks a workgroup (LDS).
    team[i] = std::max((blocks[i] + 1023) / 1024, one_slot ? (*base_team)[i] : 1u);
    team[i] = std::min(team[i], blocks[i]);
  }
  // Team sizes for the least time x in which all can end: every cloud gets the smallest team
  // that ends within x; teams hold their workgroups at once, and the clouds of one workgroup
  // share the rest (one-slot launches: every cloud holds its own).
  std::vector<RoundsTeams> choice(n);
  double lo = 0.0, hi = 1.0;
  for (size_t i = 0; i < n; ++i) {
    choice[i] = rounds_teams(specs[i], target[i], team[i], std::min(blocks[i], kMaxTeam));
    hi = std::max(hi, choice[i].us[0]);
  }
  std::vector<double> us(n);
  for (size_t i = 0; i < n; ++i) us[i] = choice[i].us[0];
  for (int it = 0; it < 24; ++it) {
    const double x = 0.5 * (lo + hi);
    uint64_t held = 0;
    double shared = 0.0;
    for (size_t i = 0; i < n; ++i) {
      const uint32_t t = choice[i].smallest(x);
      if (choice[i].team[t] > 1 || one_slot)
        held += choice[i].team[t];
      else
        shared += choice[i].us[t] / x;
    }
    if (held + (uint64_t)std::ceil(shared) <= gmax) {
      hi = x;
      for (size_t i = 0; i < n; ++i) {
        const uint32_t t = choice[i].smallest(x);
        team[i] = choice[i].team[t];
        us[i] = choice[i].us[t];
      }
    } else {
      lo = x;
    }
  }
  uint64_t total = 0;
  for (size_t i = 0; i < n; ++i) total += team[i];
  // Teams first (they form at once while the grid is free), longest first.
  std::stable_sort(order.begin(), order.end(), [&](size_t x, size_t y) {
    const bool tx = team[x] > 1, ty = team[y] > 1;
    if (tx != ty) return tx;
    return us[x] > us[y];
  });
  members = (uint32_t)total;
  if (one_slot && members > gmax)
    return fail(FPSX_ETOOBIG, "one-slot launch: more members than co-resident workgroups");
  grid = std::min(members, gmax);
  // One buffer to clear: status and claim, the teams' counters, their exchange areas.
  size_t words = 2 + (n + 1) / 2;
  std::vector<size_t> area(n, 0);
  uint32_t nbl = 1;
  for (size_t i = 0; i < n; ++i) {
    nbl = std::max(nbl, (blocks[i] + team[i] - 1) / team[i]);
    if (team[i] > grid) return fail(FPSX_ETOOBIG, "a team is larger than the co-resident grid");
    if (team[i] == 1) continue;
    area[i] = words;
    words += rounds_xchg_words(team[i], (uint32_t)dim, rounds_cap_wg(team[i]));
  }
  clear_words = words;
  shmem = rounds_shmem((uint32_t)dim, nbl);
  if (c.max_blocks(k, shmem) < (int)gmax) return fail(FPSX_ETOOBIG, "threshold rounds: LDS");
  HIP_TRY(d_clear.reserve(words * sizeof(uint64_t)));
  table_words = (n * sizeof(RoundsParams) + members * sizeof(uint32_t) + 7) / 8;
  HIP_TRY(d_tables.reserve(table_words * sizeof(uint64_t)));
  if (one_slot) {
    const size_t need = kPinnedHead + table_words * sizeof(uint64_t);
    if (need > pinned_cap) {
      if (pinned) (void)hipHostFree(pinned);
      pinned = nullptr;
      pinned_cap = 0;
      HIP_TRY(hipHostMalloc((void **)&pinned, 2 * need, hipHostMallocDefault));
      pinned_cap = 2 * need;
    }
    std::memset(pinned, 0, need);
  } else {
    host.assign(table_words * sizeof(uint64_t), 0);
  }
  RoundsParams *tab = (RoundsParams *)(one_slot ? pinned + kPinnedHead : host.data());
  uint32_t *slot = (uint32_t *)(tab + n);
  uint64_t *cl = (uint64_t *)d_clear.p;
  uint32_t at = 0;
  for (size_t o = 0; o < n; ++o) {
    const size_t i = order[o];
    const JobSpec &s = specs[i];
    RoundsParams &r = tab[o];
    r.fps.pts = b.pts + s.pt_off;
    r.fps.ld = s.ld;
    r.fps.sp = s.sp;
    r.fps.n = s.n;
    r.fps.m = s.m;
    r.fps.n_starts = 1;
    r.fps.dim = (uint32_t)dim;
    r.fps.out = b.out + s.out_off;
    r.fps.xchg = cl + area[i];
    r.fps.status = (uint32_t *)d_clear.p;
    r.fps.dmin = b.state + s.state_off;
    r.fps.init = INFINITY;
    r.fps.spin_ticks = c.spin_ticks;
    r.rec = (const float4 *)(b.sorted + s.sorted_off);
    r.rest = b.rest ? b.rest + s.perm_off : nullptr;
    r.nblocks = blocks[i];
    r.cap_wg = rounds_cap_wg(team[i]);
    r.target = target[i];
    r.s_begin = s.s_begin;
    r.s_end = s.s_end;
    r.carry = (uint32_t *)(r.fps.dmin + s.n);
    r.start = s.start;
    r.team = team[i];
    r.member_base = at;
    r.ready = (uint32_t *)(cl + 2) + o;
    r.form_ticks = one_slot ? c.spin_ticks * 5 : c.spin_ticks;
    r.host_status = one_slot ? (uint32_t *)pinned : nullptr;
    for (uint32_t q = 0; q < team[i]; ++q) slot[at++] = (uint32_t)o;
  }
  if (!one_slot)
    HIP_TRY(hipMemcpy(d_tables.p, host.data(), host.size(), hipMemcpyHostToDevice));
  jobs.table = (const RoundsParams *)d_tables.p;
  jobs.member_job = (const uint32_t *)(jobs.table + n);
  jobs.members = members;
  jobs.claim = (uint32_t *)(cl + 1);
  jobs.team_ticks = c.spin_ticks * 5;
  jobs.one_slot = one_slot ? 1u : 0u;
  return FPSX_OK;
}

int RoundsRun::enqueue(hipStream_t st, hipEvent_t begin, hipEvent_t end) {
  if (jobs.one_slot) {
    const size_t w = std::max(clear_words, table_words);
    hipLaunchKernelGGL(stage_jobs, dim3((unsigned)std::min<size_t>(1024, (w + 255) / 256)),
                       dim3(256), 0, st, (const uint64_t *)(pinned + kPinnedHead),
                       (uint64_t *)d_tables.p, table_words, (uint64_t *)d_clear.p, clear_words);
    HIP_TRY(hipGetLastError());
  } else {
    HIP_TRY(launch_fill_u64((uint64_t *)d_clear.p, clear_words, 0, st));
  }
  void *args[] = {(void *)&jobs};
  if (end) {
    HIP_TRY(hipExtLaunchKernel(k->fn, dim3(grid), dim3(k->block), args, shmem, st, begin, end, 0));
  } else {
    HIP_TRY(hipLaunchKernel(k->fn, dim3(grid), dim3(k->block), args, shmem, st));
  }
  return FPSX_OK;
}

}  // namespace fpsx

using namespace fpsx;

// ---------------------------------------------------------------------------
// Batch object
// ---------------------------------------------------------------------------
struct fpsx_batch {
  Ctx *ctx = nullptr;
  int dim = 0;
  size_t n_clouds = 0;
  BatchRun run;
  // Pruned kernel (fps_batch_pp): every cloud in spatial order, cloud c's
  // coordinates at sorted + 3 * offsets[c] (SoA, ld = its size) and original
  // indices at perm + offsets[c]; blocks of `order_block` positions.
  DevBuf sorted, perm;
  SpatialScratch *spatial = nullptr;
  uint32_t order_block = 0;
  std::vector<uint64_t> offsets;
  // Threshold rounds: records of cloud c at rec + 4 * offsets[c], coordinates beyond three
  // at rest, min-distances of clouds too large for registers in state.
  RoundsRun rounds;
  bool use_rounds = false;
  DevBuf rec, rest, state;
  DevBuf d_order;  // but for 3-D: the pieces that every run puts in spatial order
  uint32_t order_jobs = 0;
  RoundsOrderScratch *rorder = nullptr;
  bool fallback = false;  // no batch kernel for this dimension or cloud size: one launch per cloud
  std::vector<JobSpec> specs;
  const float *d_pts = nullptr;
  uint64_t ld = 0;
  uint64_t *d_out = nullptr;
  hipStream_t capture_stream = nullptr;
  hipGraph_t graph = nullptr;
  hipGraphExec_t exec = nullptr;
  // What the rounds took, where they do not serve.
  void drop_rounds() {
    for (DevBuf *m : {&rec, &rest, &state, &d_order, &rounds.d_tables, &rounds.d_clear}) m->free();
    delete_rounds_order_scratch(rorder);
    rorder = nullptr;
    order_jobs = 0;
  }
  void *status_word() const { return use_rounds ? rounds.d_clear.p : run.d_status.p; }
};

static int validate_batch(const uint64_t *offsets, size_t n_clouds, const uint64_t *n_samples,
                          const uint64_t *start_idx, uint64_t ld, std::vector<JobSpec> &specs) {
  if (!offsets || !n_samples || !start_idx || n_clouds == 0)
    return fail(FPSX_EINVAL, "empty batch or null pointer");
  specs.resize(n_clouds);
  uint64_t out_off = 0;
  for (size_t c = 0; c < n_clouds; ++c) {
    if (offsets[c + 1] < offsets[c]) return fail(FPSX_EINVAL, "offsets must not decrease");
    const uint64_t n = offsets[c + 1] - offsets[c];
    if (n == 0) return fail(FPSX_EINVAL, "cloud " + std::to_string(c) + " is empty");
    if (n >= (uint64_t(1) << 31)) return fail(FPSX_ETOOBIG, "cloud too large");
    if (n_samples[c] == 0 || n_samples[c] > n)
      return fail(FPSX_EINVAL, "cloud " + std::to_string(c) + ": n_samples must be in [1, n]");
    if (start_idx[c] >= n)
      return fail(FPSX_EBADSTART, "cloud " + std::to_string(c) + ": start index out of range");
    JobSpec &s = specs[c];
    s.pt_off = offsets[c];
    s.ld = ld;
    s.out_off = out_off;
    s.state_off = 0;
    s.start = start_idx[c];
    s.n = (uint32_t)n;
    s.m = (uint32_t)n_samples[c];
    s.s_begin = 0;
    s.s_end = s.m;
    out_off += n_samples[c];
  }
  return FPSX_OK;
}

// Put every cloud in spatial order with blocks of `block` positions (once
// per block size), on the context's stream.  Caller holds the context lock.
static int batch_order(fpsx_batch *b, uint32_t block) {
  if (b->order_block == block) return FPSX_OK;
  const uint64_t total = b->offsets.back();
  uint32_t nmax = 0;
  for (auto &s : b->specs) nmax = std::max(nmax, s.n);
  HIP_TRY(b->sorted.reserve(total * 3 * sizeof(float)));
  HIP_TRY(b->perm.reserve(total * sizeof(uint32_t)));
  if (!b->spatial) b->spatial = new_spatial_scratch();
  int rc = spatial_reserve(*b->spatial, nmax, block);
  if (rc) return rc;
  hipStream_t st = b->ctx->stream;
  for (size_t c = 0; c < b->n_clouds; ++c) {
    const uint64_t off = b->offsets[c];
    rc = spatial_order(b->d_pts + off, 1, b->ld, b->specs[c].n, block,
                       (float *)b->sorted.p + 3 * off, (uint32_t *)b->perm.p + off, *b->spatial, st);
    if (rc) return rc;
  }
  HIP_TRY(hipStreamSynchronize(st));
  b->order_block = block;
  return FPSX_OK;
}

// The threshold rounds for this batch: order its clouds, build the tables.  ETOOBIG where
// some cloud is beyond a team of the pass kernels too.  Caller holds the context lock.
//   3-D clouds are put in spatial order here, as for the pruned kernels.  For other dimensions
//   nothing reads the caller's points before a run does, at its place in the stream: each run
//   orders them anew, in one launch and so in pieces of 8192 (batch_enqueue).  Two dimensions,
//   us a run so, without any order, and with a whole order made here: 48 clouds of 1024 to 16384
//   points 661, 853 and 636; 16 of 20 K to 200 K 2152, 4308 and 1678.
static int batch_prepare_rounds(fpsx_batch *b) {
  Ctx &c = *b->ctx;
  const uint64_t total = b->offsets.back();
  const uint64_t more = b->dim > 3 ? (uint64_t)b->dim - 3 : 0;
  uint32_t nmax = 0;
  for (auto &s : b->specs) nmax = std::max(nmax, s.n);
  if (nmax > kMaxTeam * 16384u) return fail(FPSX_ETOOBIG, "a cloud exceeds a team's capacity");
  HIP_TRY(b->rec.reserve(total * sizeof(float4)));
  if (more) HIP_TRY(b->rest.reserve(total * more * sizeof(float)));
  // (n + 4 floats a cloud, 16-byte aligned)
  std::vector<JobSpec> specs = b->specs;
  uint64_t at = 0;
  for (size_t i = 0; i < b->n_clouds; ++i) {
    specs[i].sorted_off = 4 * b->offsets[i];
    specs[i].perm_off = more * b->offsets[i];
    specs[i].state_off = at;
    at += ((uint64_t)specs[i].n + 7) / 4 * 4;
  }
  HIP_TRY(b->state.reserve(at * sizeof(float)));
  int rc = FPSX_OK;
  if (b->dim == 3) {
    if (!b->rorder) b->rorder = new_rounds_order_scratch();
    rc = rounds_order_reserve(*b->rorder, nmax);
    for (size_t i = 0; i < b->n_clouds && !rc; ++i)
      rc = rounds_order(b->d_pts + specs[i].pt_off, 1, b->ld, specs[i].n, 3,
                        (float4 *)b->rec.p + b->offsets[i], nullptr, *b->rorder, c.stream);
    if (rc) return rc;
    HIP_TRY(hipStreamSynchronize(c.stream));
  } else {
    std::vector<RoundsOrderJob> jobs;
    for (size_t i = 0; i < b->n_clouds; ++i)
      rounds_order_pieces(b->d_pts + specs[i].pt_off, 1, b->ld, specs[i].n, (uint32_t)b->dim,
                          (float4 *)b->rec.p + b->offsets[i],
                          more ? (float *)b->rest.p + specs[i].perm_off : nullptr, jobs);
    b->order_jobs = (uint32_t)jobs.size();
    HIP_TRY(b->d_order.reserve(jobs.size() * sizeof(RoundsOrderJob)));
    HIP_TRY(hipMemcpy(b->d_order.p, jobs.data(), jobs.size() * sizeof(RoundsOrderJob),
                      hipMemcpyHostToDevice));
  }
  const RoundsBases bases = {b->d_pts, b->d_out, (float *)b->state.p, (const float *)b->rec.p,
                             (const float *)b->rest.p};
  return b->rounds.prepare(c, b->dim, specs, bases);
}

// One run's launches (graph-capturable).
static int batch_enqueue(fpsx_batch *b, hipStream_t st) {
  if (!b->use_rounds) return b->run.enqueue(st);
  if (b->order_jobs)
    HIP_TRY(launch_order_pieces((const RoundsOrderJob *)b->d_order.p, b->order_jobs, st));
  return b->rounds.enqueue(st);
}

static int batch_prepare_kernel(fpsx_batch *b, const KernelEntry *k, bool pruned) {
  std::vector<BatchJob> jobs;
  std::vector<uint32_t> mj;
  uint32_t areas = 0;
  if (pruned) {
    for (size_t c = 0; c < b->n_clouds; ++c) {
      b->specs[c].sorted_off = 3 * b->offsets[c];
      b->specs[c].perm_off = b->offsets[c];
    }
  }
  int rc = build_jobs(b->specs.data(), b->specs.size(), k, 0, jobs, mj, &areas, pruned);
  if (rc) return rc;
  if (pruned) {
    rc = batch_order(b, (uint32_t)(64 * k->ppt));
    if (rc) return rc;
    return b->run.prepare(*b->ctx, k, jobs, mj, areas, b->d_pts, b->d_out, nullptr,
                          (const float *)b->sorted.p, (const uint32_t *)b->perm.p, false);
  }
  return b->run.prepare(*b->ctx, k, jobs, mj, areas, b->d_pts, b->d_out, nullptr);
}

// An internal flag of fpsx_batch_create: the batch is run once.
constexpr int kBatchOnce = 1 << 16;

// Whether the pass kernels run a 3-D batch faster: the first picks of a cloud come one or two a
// round.  Passes and rounds, us a run: 512 clouds of 1000 points 72 and 107 at 8 picks, 134 and
// 157 at 32, 218 and 194 at 64; 64 of 16000 124 and 168 at 32, 180 and 205 at 64; 64 of 60000 358
// and 439 at 64, 585 and 519 at 128.  Run once, with the order made for it, rounds are ahead from
// 32 picks too (8 clouds of 16000 from host memory 1097 and 917).
static bool few_picks(const std::vector<JobSpec> &specs) {
  uint32_t m = 0, n = 0;
  for (auto &s : specs) {
    m = std::max(m, s.m);
    n = std::max(n, s.n);
  }
  return m < (n > 8192 ? 96u : 64u);
}

FPSX_EXPORT int fpsx_batch_create(const float *d_points, size_t ld, size_t dim,
                                  const uint64_t *offsets, size_t n_clouds,
                                  const uint64_t *n_samples, const uint64_t *start_idx,
                                  uint64_t *d_out, int flags, fpsx_batch **out) {
  if (!out) return fail(FPSX_EINVAL, "null output handle");
  *out = nullptr;
  if (dim == 0) return fail(FPSX_EBADDIM, "dim must be >= 1");
  if (!d_points || !d_out) return fail(FPSX_EINVAL, "null pointer argument");
  struct Destroy {
    void operator()(fpsx_batch *p) const { fpsx_batch_destroy(p); }
  };
  std::unique_ptr<fpsx_batch, Destroy> b(new fpsx_batch());
  int rc = validate_batch(offsets, n_clouds, n_samples, start_idx, ld, b->specs);
  if (rc) return rc;
  if (ld < offsets[n_clouds]) return fail(FPSX_EINVAL, "ld must be >= the total point count");
  rc = get_ctx(&b->ctx);
  if (rc) return rc;
  b->dim = (int)dim;
  b->n_clouds = n_clouds;
  b->d_pts = d_points;
  b->ld = ld;
  b->d_out = d_out;
  b->offsets.assign(offsets, offsets + n_clouds + 1);
  Ctx &c = *b->ctx;
  std::lock_guard<std::mutex> lk(c.mu);

  // Candidates: 3-D batches first the pruned paired kernels (spatial order,
  // wave boxes, two picks per team exchange; FPSX_BATCH_PLAIN=1 leaves them
  // out), then the plain batch kernels of the dimension.
  struct Cand {
    const KernelEntry *k;
    bool pruned;
  };
  std::vector<Cand> cands;
  const char *plain = std::getenv("FPSX_BATCH_PLAIN");
  // Threshold rounds unless a pass kernel is asked for by name; the tuner times them too.
  bool rounds = rounds_jobs_kernel((int)dim) != nullptr;
  for (const char *name : {"FPSX_BATCH_SHAPE", "FPSX_BATCH_PLAIN", "FPSX_BATCH_NO_PAIR", "FPSX_NO_ROUNDS"}) {
    const char *v = std::getenv(name);
    if (v && *v && std::strcmp(v, "0") != 0) rounds = false;
  }
  if (dim == 3 && !(flags & (FPSX_BATCH_AUTOTUNE | kBatchOnce)) && few_picks(b->specs)) rounds = false;
  float rounds_ms = 1e30f;
  if (rounds) {
    rc = batch_prepare_rounds(b.get());
    if (rc != FPSX_OK && rc != FPSX_ETOOBIG && rc != FPSX_ENOMEM) return rc;
    rounds = rc == FPSX_OK;
    if (!rounds) b->drop_rounds();
  }
  if (rounds && (flags & FPSX_BATCH_AUTOTUNE)) {
    hipEvent_t e0, e1;
    HIP_TRY(hipEventCreate(&e0));
    HIP_TRY(hipEventCreate(&e1));
    HIP_TRY(hipEventRecord(e0, c.stream));
    b->use_rounds = true;
    rc = batch_enqueue(b.get(), c.stream);
    if (rc) return rc;
    HIP_TRY(hipEventRecord(e1, c.stream));
    HIP_TRY(hipEventSynchronize(e1));
    float ms = 0.0f;
    HIP_TRY(hipEventElapsedTime(&ms, e0, e1));
    (void)hipEventDestroy(e0);  // timing events only
    (void)hipEventDestroy(e1);
    HIP_TRY(hipMemcpy(c.host_status, b->rounds.status(), sizeof(uint32_t), hipMemcpyDeviceToHost));
    if (*c.host_status == 0) rounds_ms = ms;  // a run that gave up is not fast
  }
  if (dim == 3 && !(plain && plain[0] == '1')) {
    for (int ppt : {8, 16, 4}) {
      const KernelEntry *k = batch_pp_kernel(1024, ppt, false);
      if (k) cands.push_back({k, true});
    }
  }
  size_t cnt;
  const KernelEntry *t = batch_table(&cnt);
  for (size_t i = 0; i < cnt; ++i)
    if (t[i].dim == (int)dim) cands.push_back({&t[i], false});
  if (cands.empty() && !rounds) {
    b->fallback = true;
    *out = b.release();
    return FPSX_OK;
  }
  const KernelEntry *chosen = nullptr;
  bool chosen_pruned = false;
  const char *env = std::getenv("FPSX_BATCH_SHAPE");
  int eb = 0, ep = 0;
  if (env && std::sscanf(env, "pp:%d:%d", &eb, &ep) == 2) {
    chosen = batch_pp_kernel(eb, ep, false);
    chosen_pruned = chosen != nullptr && dim == 3;
    if (!chosen_pruned) chosen = nullptr;
  } else if (env && std::sscanf(env, "%d:%d", &eb, &ep) == 2) {
    chosen = find_batch((int)dim, eb, ep);
  }
  if (!chosen && (flags & FPSX_BATCH_AUTOTUNE)) {
    // Time one launch of every shape that can hold the batch; keep the fastest.
    hipEvent_t e0, e1;
    HIP_TRY(hipEventCreate(&e0));
    HIP_TRY(hipEventCreate(&e1));
    float best = rounds_ms;
    for (const Cand &cd : cands) {
      const KernelEntry *k = cd.k;
      if (batch_prepare_kernel(b.get(), k, cd.pruned) != FPSX_OK) continue;
      HIP_TRY(hipEventRecord(e0, c.stream));
      if (b->run.enqueue(c.stream) != FPSX_OK) continue;
      HIP_TRY(hipEventRecord(e1, c.stream));
      HIP_TRY(hipEventSynchronize(e1));
      float ms = 0;
      HIP_TRY(hipEventElapsedTime(&ms, e0, e1));
      HIP_TRY(hipMemcpy(c.host_status, b->run.d_status.p, sizeof(uint32_t), hipMemcpyDeviceToHost));
      if (*c.host_status == 0 && ms < best) {
        best = ms;
        chosen = k;
        chosen_pruned = cd.pruned;
      }
    }
    (void)hipEventDestroy(e0);  // timing events only
    (void)hipEventDestroy(e1);
  }
  b->use_rounds = rounds && !chosen;
  if (!chosen && !b->use_rounds) {
    // Heuristic: the first pruned kernel whose teams hold every cloud; else
    // the smallest plain per-workgroup capacity that still fits every cloud
    // in a team the grid can hold (short reduction chains for small clouds),
    // falling back to larger shapes.
    uint32_t nmax = 0;
    for (auto &s : b->specs) nmax = std::max(nmax, s.n);
    for (const Cand &cd : cands) {
      if (!cd.pruned) continue;
      const uint32_t cap = (uint32_t)(cd.k->block * cd.k->ppt);
      if ((nmax + cap - 1) / cap <= kMaxTeam) {
        chosen = cd.k;
        chosen_pruned = true;
        break;
      }
    }
    static const int kOrder[][2] = {{256, 16}, {1024, 16}, {256, 32}, {1024, 8}, {256, 8}, {256, 4}};
    for (auto &sh : kOrder) {
      if (chosen) break;
      const KernelEntry *k = find_batch((int)dim, sh[0], sh[1]);
      if (!k) continue;
      if ((nmax + (uint32_t)(sh[0] * sh[1]) - 1) / (uint32_t)(sh[0] * sh[1]) > 8 && sh[0] * sh[1] < 16384)
        continue;
      chosen = k;
    }
    if (!chosen) {
      chosen = cands.back().k;
      chosen_pruned = cands.back().pruned;
    }
  }
  rc = b->use_rounds ? FPSX_OK : batch_prepare_kernel(b.get(), chosen, chosen_pruned);
  if (rc == FPSX_ETOOBIG) {
    // Some cloud needs more workgroups than a team may have: every cloud
    // gets a planned launch of its own (the single-cloud kernels have no
    // such limit).
    b->fallback = true;
    *out = b.release();
    return FPSX_OK;
  }
  if (rc) return rc;
  // The status until the first run.
  const uint32_t ok = 0;
  HIP_TRY(hipMemcpy(b->status_word(), &ok, sizeof(ok), hipMemcpyHostToDevice));
  if (flags & FPSX_BATCH_GRAPH) {
    HIP_TRY(hipStreamCreateWithFlags(&b->capture_stream, hipStreamNonBlocking));
    HIP_TRY(hipStreamBeginCapture(b->capture_stream, hipStreamCaptureModeThreadLocal));
    rc = batch_enqueue(b.get(), b->capture_stream);
    hipGraph_t g = nullptr;
    hipError_t e = hipStreamEndCapture(b->capture_stream, &g);
    if (rc) return rc;
    if (e != hipSuccess) return hip_err(e, "hipStreamEndCapture");
    b->graph = g;
    HIP_TRY(hipGraphInstantiate(&b->exec, g, nullptr, nullptr, 0));
  }
  *out = b.release();
  return FPSX_OK;
}

FPSX_EXPORT int fpsx_batch_run(fpsx_batch *b, void *stream) {
  if (!b) return fail(FPSX_EINVAL, "null batch");
  Ctx &c = *b->ctx;
  std::lock_guard<std::mutex> lk(c.mu);
  hipStream_t st = stream ? (hipStream_t)stream : c.stream;
  if (b->fallback) {
    // No batch kernel for this dimension or cloud size: one planned launch
    // per cloud.  Every launch clears the context's status word, so each
    // one's status is folded into the batch's own word, which the batch
    // status then reports (a failure in any cloud, not only the last).
    HIP_TRY(b->run.d_status.reserve(sizeof(uint64_t)));
    int rc = scratch_acquire(c, st);
    if (rc) return rc;
    HIP_TRY(launch_fill_u64((uint64_t *)b->run.d_status.p, 1, 0, st));
    HIP_TRY(c.starts.reserve(b->specs.size() * sizeof(uint64_t)));
    std::vector<uint64_t> starts(b->specs.size());
    for (size_t i = 0; i < starts.size(); ++i) starts[i] = b->specs[i].start;
    HIP_TRY(hipMemcpyAsync(c.starts.p, starts.data(), starts.size() * sizeof(uint64_t),
                           hipMemcpyHostToDevice, st));
    for (size_t i = 0; i < b->specs.size(); ++i) {
      const JobSpec &s = b->specs[i];
      Plan p;
      rc = plan_call(c, s.n, b->dim, kTieHighest, s.m, p);
      if (rc) return rc;
      rc = launch_fps(c, p, b->d_pts + s.pt_off, 1, b->ld, s.n, b->dim, s.m,
                      (const uint64_t *)c.starts.p + i, 1, b->d_out + s.out_off, nullptr,
                      INFINITY, st);
      if (rc) return rc;
      HIP_TRY(launch_or_u32((const uint32_t *)c.status.p, (uint32_t *)b->run.d_status.p, st));
    }
    return scratch_release(c, st);
  }
  if (b->exec) {
    HIP_TRY(hipGraphLaunch(b->exec, st));
    return FPSX_OK;
  }
  return batch_enqueue(b, st);
}

FPSX_EXPORT int fpsx_batch_status(fpsx_batch *b, void *stream) {
  if (!b) return fail(FPSX_EINVAL, "null batch");
  Ctx &c = *b->ctx;
  std::lock_guard<std::mutex> lk(c.mu);
  hipStream_t st = stream ? (hipStream_t)stream : c.stream;
  HIP_TRY(hipStreamSynchronize(st));
  if (!b->status_word()) return FPSX_OK;  // never run
  HIP_TRY(hipMemcpy(c.host_status, b->status_word(), sizeof(uint32_t), hipMemcpyDeviceToHost));
  return status_code(*c.host_status);
}

FPSX_EXPORT int fpsx_batch_info(fpsx_batch *b, int *block, int *ppt, int *grid, int *members,
                                int *graph) {
  if (!b) return fail(FPSX_EINVAL, "null batch");
  const KernelEntry *k = b->fallback ? nullptr : b->use_rounds ? b->rounds.k : b->run.k;
  if (block) *block = k ? k->block : 0;
  if (ppt) *ppt = k ? k->ppt : 0;
  if (grid) *grid = !k ? 0 : (int)(b->use_rounds ? b->rounds.grid : b->run.grid);
  if (members) *members = !k ? 0 : (int)(b->use_rounds ? b->rounds.members : b->run.members);
  if (graph) *graph = b->exec != nullptr;
  return FPSX_OK;
}

FPSX_EXPORT void fpsx_batch_destroy(fpsx_batch *b) {
  if (!b) return;
  // Release path: a failed destroy leaves nothing for the caller to do.
  if (b->exec) (void)hipGraphExecDestroy(b->exec);
  if (b->graph) (void)hipGraphDestroy(b->graph);
  if (b->capture_stream) (void)hipStreamDestroy(b->capture_stream);
  b->sorted.free();
  b->perm.free();
  b->drop_rounds();
  delete_spatial_scratch(b->spatial);
  delete b;
}

FPSX_EXPORT int fpsx_fps_batch(const float *points, size_t dim, const uint64_t *offsets,
                               size_t n_clouds, const uint64_t *n_samples,
                               const uint64_t *start_idx, uint64_t *out) {
  if (dim == 0) return fail(FPSX_EBADDIM, "dim must be >= 1");
  if (!points || !out) return fail(FPSX_EINVAL, "null pointer argument");
  std::vector<JobSpec> specs;
  int rc = validate_batch(offsets, n_clouds, n_samples, start_idx, offsets[n_clouds], specs);
  if (rc) return rc;
  const size_t total = offsets[n_clouds];
  size_t total_m = 0;
  for (size_t c = 0; c < n_clouds; ++c) total_m += n_samples[c];
  Ctx *cp = nullptr;
  rc = get_ctx(&cp);
  if (rc) return rc;
  DevBuf rows, soa, dout;
  HIP_TRY(rows.reserve(total * dim * sizeof(float)));
  HIP_TRY(soa.reserve(total * dim * sizeof(float)));
  HIP_TRY(dout.reserve(total_m * sizeof(uint64_t)));
  {
    std::lock_guard<std::mutex> lk(cp->mu);
    HIP_TRY(hipMemcpyAsync(rows.p, points, total * dim * sizeof(float), hipMemcpyHostToDevice,
                           cp->stream));
    HIP_TRY(launch_strided_to_soa((const float *)rows.p, dim, 1, (float *)soa.p, (uint32_t)total,
                                  (uint32_t)dim, total, cp->stream));
    HIP_TRY(hipStreamSynchronize(cp->stream));
  }
  fpsx_batch *b = nullptr;
  rc = fpsx_batch_create((const float *)soa.p, total, dim, offsets, n_clouds, n_samples, start_idx,
                         (uint64_t *)dout.p, kBatchOnce, &b);
  if (rc == FPSX_OK) rc = fpsx_batch_run(b, nullptr);
  if (rc == FPSX_OK) rc = fpsx_batch_status(b, nullptr);
  if (rc == FPSX_OK) {
    hipError_t e = hipMemcpy(out, dout.p, total_m * sizeof(uint64_t), hipMemcpyDeviceToHost);
    if (e != hipSuccess) rc = hip_err(e, "hipMemcpy");
  }
  fpsx_batch_destroy(b);
  rows.free();
  soa.free();
  dout.free();
  return rc;
}
