// bk_batch.hip -- batched sweeps over many independent grids.
//
// A batch holds one device table per (stencil, dtype) group and one per
// dtype for the ghost refresh.  bk_batch_set() writes the current requests
// into those tables (pinned staging, then one stream-ordered kernel that
// fetches the parts in use into HBM: 49 copies, most of empty tables, took
// 0.5 ms of a batch's set, one launch 12 us);
// bk_batch_run() launches, per tick, one persistent refresh kernel per dtype
// and one persistent sweep kernel per group -- each serving the
// concatenated work of all its requests -- optionally captured once into a
// hipGraph and replayed.  The launch grids do not depend on the table
// contents, so a captured run stays valid when the host rewrites the
// tables between runs (continuous batching).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstddef>
#include <cstring>
#include <map>
#include <memory>
#include <mutex>
#include <new>
#include <tuple>
#include <utility>

#include "bk_api.h"
#include "bk_graphs.h"
#include "bk_internal.h"

namespace bk {
int plan_fail(int code, const char *msg);
}

namespace {
// sweep groups: (stencil, dtype, schedule); the schedule of a star request
// is 0 without a plan (one brick per wave), 1 with a column plan (k-marching
// units), 2 with a quad plan (2x2 blocks of k-columns per workgroup)
constexpr int kStencils = 5, kDtypes = 3, kScheds = 3, kGroups = kStencils * kDtypes * kScheds;
static_assert(kGroups <= 64, "the non-empty groups form a 64-bit mask");
constexpr size_t kCoeffSlot = 125;  // doubles per request in the coefficient pool
// above the groups' bits of a sweep mask: two bits per dtype with the planes a
// wave of the cube's block form (0: marching form), so that a captured run's
// key tells the kernels it launches
constexpr int kPlaneBits = kGroups;
static_assert(kPlaneBits + 2 * kDtypes <= 64, "the cube's forms fit the mask");

constexpr int cube_planes(uint64_t mask, int dtype) {
  return (int)(mask >> (kPlaneBits + 2 * dtype)) & 3;
}

// Tables and coefficients lie at the same offsets of one pinned and one device
// allocation.
constexpr size_t kTableStride = (sizeof(bk::BatchTable) + 255) & ~(size_t)255;
constexpr size_t kCoeffAt = kTableStride * (kGroups + kDtypes);

// Byte ranges of the staging memory in use, in units of 16 bytes.
constexpr int kMaxRanges = 2 * (kGroups + kDtypes) + 1;
struct Ranges {
  uint32_t at[kMaxRanges], len[kMaxRanges];
};
static_assert(offsetof(bk::BatchTable, seg) % 16 == 0 && sizeof(bk::BatchSeg) % 16 == 0,
              "table parts are ranges of 16-byte units");

// Copies range blockIdx.y from the (pinned) staging memory.
__global__ __launch_bounds__(256) void fetch_ranges(const uint4 *__restrict__ from,
                                                    uint4 *__restrict__ to, const Ranges r) {
  const uint32_t at = r.at[blockIdx.y], len = r.len[blockIdx.y];
  for (uint32_t q = blockIdx.x * 256 + threadIdx.x; q < len; q += gridDim.x * 256)
    to[at + q] = from[at + q];
}

constexpr int group_of(int stencil, int dtype, int sched) {
  return (stencil * kDtypes + dtype) * kScheds + sched;
}
constexpr int dtype_of(int group) { return (group / kScheds) % kDtypes; }

using Span = std::pair<uintptr_t, uintptr_t>;  // a field's bytes

// Side streams of a run whose chains go side by side.
constexpr int kSide = 3;
}  // namespace

struct bk_batch_s {
  int device = 0;
  uint32_t max_reqs = 0;
  char *d_mem = nullptr;  // the tables and the coefficient pool
  char *h_mem = nullptr;  // their staging copy, pinned
  bk::BatchTable *d_sweep[kGroups] = {};
  bk::BatchTable *h_sweep[kGroups] = {};
  bk::BatchTable *d_ref[kDtypes] = {};
  bk::BatchTable *h_ref[kDtypes] = {};
  double *d_coeff = nullptr;
  double *h_coeff = nullptr;
  uint64_t sweep_mask = 0;  // non-empty sweep groups
  uint32_t ref_mask = 0;    // non-empty refresh tables
  hipEvent_t staged = nullptr;
  hipStream_t capture = nullptr;
  hipStream_t side[kSide] = {};  // captured runs whose groups go side by side
  hipEvent_t forked = nullptr, joined[kSide] = {};
  std::unique_ptr<Span[]> span;  // bk_batch_set's: 2 * max_reqs
  bool apart = false;  // the groups of the set may run side by side
  uint64_t bricks = 0;  // of the set's requests with sweeps left
  // captured runs keyed by (tick count, sweep groups with the cube's forms,
  // refresh groups and whether the groups go side by side); an
  // exec is destroyed only once its last launch has completed, so a caller
  // may queue the next run while the previous one is still on the device
  bk::ExecCache<std::tuple<uint32_t, uint64_t, uint32_t>> graphs{64};
  std::mutex mu;
};

namespace {

int fail(int code, const char *msg) { return bk::plan_fail(code, msg); }

int hipfail(hipError_t e, const char *what) {
  char buf[256];
  snprintf(buf, sizeof(buf), "%s: %s", what, hipGetErrorString(e));
  return fail(e == hipErrorOutOfMemory ? BK_ERR_NOMEM : BK_ERR_HIP, buf);
}

#define BKB_HIP(call)                                 \
  do {                                                \
    hipError_t e_ = (call);                           \
    if (e_ != hipSuccess) return hipfail(e_, #call);  \
  } while (0)

// No two requests' fields overlap: a field spans the bricks of its plan's
// adjacency; without a plan, whose list may hold any ids, all up to the end of
// its arena block or allocation (24 requests: 48 looked up in 6 us).
bool fields_apart(const bk_batch_req *reqs, uint32_t n, Span *span) {
  uint32_t m = 0;
  for (uint32_t r = 0; r < n; ++r) {
    const bk_batch_req &q = reqs[r];
    auto field = [&](const void *p) {
      const uintptr_t at = reinterpret_cast<uintptr_t>(p);
      return Span{at, q.plan ? at + (uintptr_t)bk::plan_view(q.plan).nbricks * q.step *
                                        bk_dtype_size(q.dtype)
                             : bk::block_end(p)};
    };
    const Span lo = field(std::min(q.d_f0, q.d_f1)), hi = field(std::max(q.d_f0, q.d_f1));
    if (lo.second > hi.first) {  // interleaved, or of one allocation
      span[m++] = {lo.first, std::max(lo.second, hi.second)};
    } else {
      span[m++] = lo;
      span[m++] = hi;
    }
  }
  std::sort(span, span + m);
  for (uint32_t i = 1; i < m; ++i)
    if (span[i].first < span[i - 1].second) return false;
  return true;
}

// Group g's sweep of tick t.
hipError_t enqueue_group(bk_batch_s *b, int g, uint32_t t, hipStream_t s) {
  const int stencil = g / (kScheds * kDtypes), dtype = dtype_of(g), sched = g % kScheds;
  if (stencil == BK_CUBE125)
    return bk::launch_cube_batched(dtype, cube_planes(b->sweep_mask, dtype), b->d_sweep[g], t, s);
  if (sched == 1) return bk::launch_star_columns_batched(stencil, dtype, b->d_sweep[g], t, s);
  if (sched == 2) return bk::launch_star_quads_batched(stencil, dtype, b->d_sweep[g], t, s);
  return bk::launch_star_batched(stencil, dtype, b->d_sweep[g], t, s);
}

// Whether a captured run forks.  Each launch gains 1 us, and another per 200
// bricks of its group and at most 10; fork and join cost 65 us, and in some
// processes, by the queues that the runtime maps its branches to, 150.  One
// stream / forked, in us: 10 groups of 8^3 bricks, 16 ticks 1312 / 721-727, 4
// ticks 356 / 250-403, 1 tick 117 / 141; 8 groups of 2^3, 16 ticks 556 /
// 471; 5 groups of 24^3, 4 ticks 1038 / 939-951.  Few launches gain less than
// several queues take from them: 3 groups of 660 bricks, 16 ticks 419 / 565, 2
// of 8^3 281 / 599.
bool forks(const bk_batch_s *b, uint32_t nticks) {
  if (!b->apart) return false;
  const int launches = __builtin_popcountll(b->sweep_mask & ((1ull << kGroups) - 1)) +
                       __builtin_popcount(b->ref_mask);
  if (launches < 5) return false;
  const double gain = 1.0 + std::min(10.0, (double)b->bricks / launches / 200.0);
  return gain * launches * nticks > 150.0;
}

// What has to run in turn, tick by tick: a type's refresh, if it has one, and
// sweep groups.
struct Chain {
  int refresh = -1;
  uint64_t groups = 0;  // mask
};

hipError_t enqueue_chain(bk_batch_s *b, const Chain &c, uint32_t t, hipStream_t s) {
  hipError_t e = hipSuccess;
  if (c.refresh >= 0) e = bk::launch_ghost_batched(c.refresh, b->d_ref[c.refresh], t, s);
  for (int g = 0; g < kGroups && e == hipSuccess; ++g)
    if (c.groups >> g & 1u) e = enqueue_group(b, g, t, s);
  return e;
}

// The streams and events of forked runs, made for the first of them.
hipError_t make_sides(bk_batch_s *b) {
  hipError_t e = hipSuccess;
  if (!b->forked) e = hipEventCreateWithFlags(&b->forked, hipEventDisableTiming);
  for (int l = 0; l < kSide && e == hipSuccess; ++l) {
    if (!b->side[l]) e = hipStreamCreateWithFlags(&b->side[l], hipStreamNonBlocking);
    if (e == hipSuccess && !b->joined[l])
      e = hipEventCreateWithFlags(&b->joined[l], hipEventDisableTiming);
  }
  return e;
}

// The launches of a run on stream s.  `fork`: chains that need nothing of each
// other (a group, or all groups of a type that refreshes ghosts) take all
// their ticks side by side, on kSide streams and s, and join once at the run's
// end.  A launch of a small group fills a fraction of
// the chip, and behind one another every tick pays every group's start and
// drain: 24 mixed requests (up to 32^3 bricks, 16 ticks, 10 groups) 1882 ->
// 1240 us side by side; with one side stream 1465 us, with seven 1831.
hipError_t enqueue_run(bk_batch_s *b, uint32_t nticks, bool fork, hipStream_t s) {
  Chain chain[kGroups];
  int nchains = 0;
  for (int d = 0; d < kDtypes; ++d)
    if (b->ref_mask >> d & 1u) chain[nchains++].refresh = d;
  const int nref = nchains;
  for (int g = 0; g < kGroups; ++g) {
    if (!(b->sweep_mask >> g & 1u)) continue;
    int c = 0;
    while (c < nref && chain[c].refresh != dtype_of(g)) ++c;
    if (c == nref) c = nchains++;
    chain[c].groups |= 1ull << g;
  }
  hipError_t e = hipSuccess;
  if (!fork || nchains < 2) {
    for (uint32_t t = 0; t < nticks; ++t)
      for (int c = 0; c < nchains && e == hipSuccess; ++c)
        e = enqueue_chain(b, chain[c], t, s);
    return e;
  }
  // chain c on side stream c, the first beyond them on s, and so on in turn
  const int sides = std::min(nchains - 1, kSide);
  e = hipEventRecord(b->forked, s);
  for (int l = 0; l < sides && e == hipSuccess; ++l)
    e = hipStreamWaitEvent(b->side[l], b->forked, 0);
  for (int c = 0; c < nchains; ++c) {
    const int l = c % (sides + 1);
    for (uint32_t t = 0; t < nticks && e == hipSuccess; ++t)
      e = enqueue_chain(b, chain[c], t, l < sides ? b->side[l] : s);
  }
  for (int l = 0; l < sides && e == hipSuccess; ++l) {
    e = hipEventRecord(b->joined[l], b->side[l]);
    if (e == hipSuccess) e = hipStreamWaitEvent(s, b->joined[l], 0);
  }
  return e;
}

}  // namespace

extern "C" {

int bk_batch_destroy(bk_batch b) {
  if (!b) return BK_OK;
  (void)b->graphs.clear();
  (void)hipFree(b->d_mem);
  (void)hipHostFree(b->h_mem);
  if (b->staged) (void)hipEventDestroy(b->staged);
  if (b->capture) (void)hipStreamDestroy(b->capture);
  if (b->forked) (void)hipEventDestroy(b->forked);
  for (int l = 0; l < kSide; ++l) {
    if (b->side[l]) (void)hipStreamDestroy(b->side[l]);
    if (b->joined[l]) (void)hipEventDestroy(b->joined[l]);
  }
  delete b;
  return BK_OK;
}

int bk_batch_create(uint32_t max_reqs, bk_batch *out) {
  if (!out) return fail(BK_ERR_ARG, "bk_batch_create: null out pointer");
  *out = nullptr;
  if (max_reqs == 0 || max_reqs > bk::kBatchMaxSegs)
    return fail(BK_ERR_ARG, "bk_batch_create: max_reqs must be in [1, 2048]");
  bk_batch_s *b = new bk_batch_s();
  b->max_reqs = max_reqs;
  b->span.reset(new (std::nothrow) Span[2 * (size_t)max_reqs]);
  (void)hipGetDevice(&b->device);
  auto cleanup = [&](int rc) {
    bk_batch_destroy(b);
    return rc;
  };
  const size_t bytes = kCoeffAt + sizeof(double) * kCoeffSlot * max_reqs + 16;
  if (!b->span || hipMalloc(&b->d_mem, bytes) != hipSuccess ||
      hipHostMalloc(&b->h_mem, bytes, hipHostMallocDefault) != hipSuccess)
    return cleanup(fail(BK_ERR_NOMEM, "bk_batch_create: table allocation failed"));
  // (a table is launched over only once a set has filled it)
  for (int g = 0; g < kGroups + kDtypes; ++g) {
    auto *d = reinterpret_cast<bk::BatchTable *>(b->d_mem + kTableStride * g);
    auto *h = reinterpret_cast<bk::BatchTable *>(b->h_mem + kTableStride * g);
    (g < kGroups ? b->d_sweep[g] : b->d_ref[g - kGroups]) = d;
    (g < kGroups ? b->h_sweep[g] : b->h_ref[g - kGroups]) = h;
  }
  b->d_coeff = reinterpret_cast<double *>(b->d_mem + kCoeffAt);
  b->h_coeff = reinterpret_cast<double *>(b->h_mem + kCoeffAt);
  if (hipEventCreateWithFlags(&b->staged, hipEventDisableTiming) != hipSuccess ||
      hipStreamCreateWithFlags(&b->capture, hipStreamNonBlocking) != hipSuccess)
    return cleanup(fail(BK_ERR_HIP, "bk_batch_create: event/stream creation failed"));
  *out = b;
  return BK_OK;
}

int bk_batch_set(bk_batch b, const bk_batch_req *reqs, uint32_t n, bk_stream stream) {
  if (!b) return fail(BK_ERR_ARG, "bk_batch_set: null batch");
  if (n && !reqs) return fail(BK_ERR_ARG, "bk_batch_set: null request array");
  if (n > b->max_reqs) return fail(BK_ERR_ARG, "bk_batch_set: more requests than max_reqs");
  hipStream_t s = static_cast<hipStream_t>(stream);
  std::lock_guard<std::mutex> lock(b->mu);
  // the staging buffers may still feed the previous set's copies
  BKB_HIP(hipEventSynchronize(b->staged));
  // validate everything before touching the tables
  for (uint32_t r = 0; r < n; ++r) {
    const bk_batch_req &q = reqs[r];
    if (bk_stencil_ncoeff(q.stencil) == 0) return fail(BK_ERR_ARG, "bk_batch_set: unknown stencil");
    if (q.dtype < 0 || q.dtype >= kDtypes) return fail(BK_ERR_ARG, "bk_batch_set: unknown dtype");
    if (!q.d_adj || !q.d_f0 || !q.d_f1 || !q.h_coeff)
      return fail(BK_ERR_ARG, "bk_batch_set: null pointer in a request");
    if (q.d_f0 == q.d_f1) return fail(BK_ERR_ARG, "bk_batch_set: a request's fields alias");
    if (q.step < 512) return fail(BK_ERR_ARG, "bk_batch_set: step smaller than a brick");
    if (q.npairs && !q.d_pairs) return fail(BK_ERR_ARG, "bk_batch_set: null pair list");
    if (q.stencil == BK_CUBE125) {
      int shape = 0;
      if (!q.plan || bk_plan_query(q.plan, nullptr, nullptr, &shape, nullptr) != BK_OK ||
          shape != BK_PLAN_QUAD)
        return fail(BK_ERR_ARG, "bk_batch_set: a cube request needs a BK_PLAN_QUAD plan");
      if (!bk::quad_offsets_fit(bk::plan_view(q.plan).nbricks, q.step))
        return fail(BK_ERR_UNSUPPORTED,
                    "bk_batch_set: the quad schedule addresses at most 2^32 input elements");
    } else if (q.plan) {
      int shape = 0;
      if (bk_plan_query(q.plan, nullptr, nullptr, &shape, nullptr) != BK_OK ||
          (shape != BK_PLAN_COLUMN && shape != BK_PLAN_QUAD))
        return fail(BK_ERR_ARG, "bk_batch_set: a star request's plan must be a BK_PLAN_COLUMN or "
                    "BK_PLAN_QUAD plan");
    } else if (q.nlist && !q.d_list) {
      return fail(BK_ERR_ARG, "bk_batch_set: null brick list");
    }
    if (q.stencil == BK_COND7 && q.cond_mode != BK_COND_REFERENCE &&
        q.cond_mode != BK_COND_THRESHOLD)
      return fail(BK_ERR_ARG, "bk_batch_set: unknown cond mode");
  }
  uint32_t count[kGroups] = {}, rcount[kDtypes] = {};
  uint64_t cube_bricks[kDtypes] = {}, bricks = 0;
  for (int g = 0; g < kGroups; ++g) b->h_sweep[g]->prefix[0] = b->h_sweep[g]->levels = 0;
  for (int d = 0; d < kDtypes; ++d) b->h_ref[d]->prefix[0] = b->h_ref[d]->levels = 0;
  for (uint32_t r = 0; r < n; ++r) {
    const bk_batch_req &q = reqs[r];
    const int sched = (q.stencil == BK_CUBE125 || !q.plan) ? 0
                      : bk::plan_view(q.plan).shape == BK_PLAN_QUAD ? 2 : 1;
    const int g = group_of(q.stencil, q.dtype, sched);
    double *slot = b->h_coeff + (size_t)r * kCoeffSlot;
    const int nc = bk_stencil_ncoeff(q.stencil);
    if (q.dtype == BK_F64) {
      for (int c = 0; c < nc; ++c) slot[c] = q.h_coeff[c];
    } else {
      float *fs = reinterpret_cast<float *>(slot);
      for (int c = 0; c < nc; ++c) fs[c] = (float)q.h_coeff[c];
    }
    bk::BatchSeg sg;
    std::memset(&sg, 0, sizeof(sg));
    sg.adj = q.d_adj;
    sg.f0 = q.d_f0;
    sg.f1 = q.d_f1;
    sg.coeff = b->d_coeff + (size_t)r * kCoeffSlot;
    sg.step = q.step;
    sg.parity = q.parity & 1u;
    sg.ticks = q.ticks;
    sg.theta = q.theta;
    sg.cond_mode = q.cond_mode;
    uint32_t nbricks = q.nlist;
    if (q.stencil == BK_CUBE125 || sched != 0) {
      const bk::PlanView P = bk::plan_view(q.plan);
      nbricks = P.ncovered;
      sg.items = P.anchor;
      sg.len = P.len;
      sg.mask = P.mask;
      sg.nitems = P.nunits;
      sg.kcol = P.kcol;
      b->h_sweep[g]->levels = std::max(b->h_sweep[g]->levels, P.longest);
      if (q.stencil == BK_CUBE125) cube_bricks[q.dtype] += nbricks;
    } else {
      sg.items = q.d_list;
      sg.nitems = q.nlist;
    }
    if (q.ticks) bricks += nbricks;
    bk::BatchTable *t = b->h_sweep[g];
    t->seg[count[g]] = sg;
    t->prefix[count[g] + 1] = t->prefix[count[g]] + sg.nitems;
    ++count[g];
    if (q.npairs) {
      bk::BatchTable *rt = b->h_ref[q.dtype];
      bk::BatchSeg rs = sg;
      rs.items = q.d_pairs;
      rs.len = rs.mask = nullptr;
      rs.nitems = q.npairs;
      rt->seg[rcount[q.dtype]] = rs;
      rt->prefix[rcount[q.dtype] + 1] = rt->prefix[rcount[q.dtype]] + q.npairs;
      ++rcount[q.dtype];
    }
  }
  b->sweep_mask = 0;
  b->ref_mask = 0;
  Ranges ranges;
  uint32_t nranges = 0, longest = 0;
  auto add = [&](size_t at, size_t bytes) {
    const uint32_t n = (uint32_t)((bytes + 15) / 16);
    ranges.at[nranges] = (uint32_t)(at / 16);
    ranges.len[nranges++] = n;
    longest = std::max(longest, n);
  };
  auto add_table = [&](int slot, const bk::BatchTable *t) {
    add(kTableStride * slot, offsetof(bk::BatchTable, prefix) + 4 * ((size_t)t->nsegs + 1));
    add(kTableStride * slot + offsetof(bk::BatchTable, seg), sizeof(bk::BatchSeg) * t->nsegs);
  };
  for (int g = 0; g < kGroups; ++g) {
    bk::BatchTable *t = b->h_sweep[g];
    t->nsegs = count[g];
    if (!count[g] || !t->prefix[count[g]]) continue;  // never launched
    b->sweep_mask |= 1ull << g;
    add_table(g, t);
  }
  for (int d = 0; d < kDtypes; ++d) {
    bk::BatchTable *t = b->h_ref[d];
    t->nsegs = rcount[d];
    if (cube_bricks[d])
      b->sweep_mask |= (uint64_t)bk::cube_batched_planes(d, cube_bricks[d])
                       << (kPlaneBits + 2 * d);
    if (!rcount[d] || !t->prefix[rcount[d]]) continue;
    b->ref_mask |= 1u << d;
    add_table(kGroups + d, t);
  }
  b->apart = fields_apart(reqs, n, b->span.get());
  b->bricks = bricks;
  if (n) add(kCoeffAt, sizeof(double) * kCoeffSlot * n);
  if (nranges) {
    hipLaunchKernelGGL(fetch_ranges, dim3((longest + 255) / 256, nranges), dim3(256), 0, s,
                       reinterpret_cast<const uint4 *>(b->h_mem),
                       reinterpret_cast<uint4 *>(b->d_mem), ranges);
    BKB_HIP(hipGetLastError());
  }
  BKB_HIP(hipEventRecord(b->staged, s));
  return BK_OK;
}

int bk_batch_run(bk_batch b, uint32_t nticks, int use_graph, bk_stream stream) {
  if (!b) return fail(BK_ERR_ARG, "bk_batch_run: null batch");
  if (nticks == 0) return BK_OK;
  hipStream_t s = static_cast<hipStream_t>(stream);
  std::lock_guard<std::mutex> lock(b->mu);
  if (!use_graph) {
    BKB_HIP(enqueue_run(b, nticks, false, s));
    return BK_OK;
  }
  const bool fork = forks(b, nticks);
  const std::tuple<uint32_t, uint64_t, uint32_t> key{
      nticks, b->sweep_mask, b->ref_mask | (fork ? 1u << kDtypes : 0u)};
  if (!b->graphs.find(key)) {
    if (fork) BKB_HIP(make_sides(b));
    BKB_HIP(hipStreamBeginCapture(b->capture, hipStreamCaptureModeThreadLocal));
    hipError_t e = enqueue_run(b, nticks, fork, b->capture);
    hipGraph_t g = nullptr;
    hipError_t e2 = hipStreamEndCapture(b->capture, &g);
    if (e != hipSuccess) {
      if (g) (void)hipGraphDestroy(g);
      return hipfail(e, "capture of batched run");
    }
    if (e2 != hipSuccess) return hipfail(e2, "hipStreamEndCapture");
    hipGraphExec_t ge = nullptr;
    e = hipGraphInstantiate(&ge, g, nullptr, nullptr, 0);
    (void)hipGraphDestroy(g);
    if (e != hipSuccess) return hipfail(e, "hipGraphInstantiate");
    BKB_HIP(b->graphs.insert(key, ge));
  }
  BKB_HIP(b->graphs.launch(key, s));
  return BK_OK;
}

}  // extern "C"
