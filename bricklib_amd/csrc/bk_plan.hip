// bk_plan.hip -- execution plans: a schedule for sweeping a set of bricks.
//
// A plan groups the bricks of a list into units a single wave can march
// through along k:
//   BK_PLAN_COLUMN  unit = up to kcol bricks b, adj[b][22], adj[adj[b][22]][22] ...
//   BK_PLAN_QUAD    unit = up to kcol levels of a 2x2 block of columns:
//                   members m0 = anchor, m1 = adj[m0][14] (i+1),
//                   m2 = adj[m0][16] (j+1), m3 = adj[m1][16]; the next level's
//                   anchor is adj[anchor][22] (k+1).
// Each (unit, level) carries a mask of the members to store; a member not
// in the list, or already covered, is computed but not stored.  Every
// listed brick is stored exactly once.  Units are emitted in the order of
// their first brick in the list, so a grid-ordered list gives spatially
// adjacent units adjacent indices (and so the same XCD).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <array>
#include <atomic>
#include <cstring>
#include <new>
#include <map>
#include <mutex>
#include <string>
#include <vector>

#include "bk_api.h"
#include "bk_internal.h"

namespace bk {
int plan_fail(int code, const char *msg);
void graphs_forget_plan(uint64_t plan_id);
}

struct bk_plan_s {
  int shape = 1;
  uint32_t kcol = 1;
  uint32_t nunits = 0;
  uint32_t longest = 0;  // levels of the longest unit
  uint32_t ncovered = 0;
  uint32_t *d_arrays = nullptr;  // one allocation holding the arrays below
  uint32_t *d_anchor = nullptr;  // [nunits] level-0 anchor
  uint32_t *d_len = nullptr;     // [nunits] levels in the unit
  uint32_t *d_mask = nullptr;    // [nunits * kcol] member store mask per level
  uint32_t *d_flat = nullptr;    // [ncovered] covered bricks in plan order
  uint32_t *d_start = nullptr;   // [nunits] offset of each unit's bricks in d_flat
  uint32_t nbricks = 0;          // bricks of the adjacency the plan was built on
  int device = 0;
  uint64_t id = 0;               // unique per plan for the process's lifetime (never 0)
  std::vector<bool> covered;     // [nbricks] the covered bricks
  // periodic box (bk_plan_set_box): brick ids in grid order, in HBM
  // (published last: a sequence of another thread may be reading the plan)
  std::atomic<uint32_t *> d_box{nullptr};
  std::mutex box_mu;  // one declaration at a time
  uint32_t *d_box_adj = nullptr;  // its wrapped adjacency, behind d_box
  uint32_t *d_box_holds = nullptr;  // [nbricks] the box brick each holds the values of, or kNone
  uint32_t *d_box_seen = nullptr;   // [nbricks] stamps of bk_plan_bind_box, then its three counts
  uint32_t box_stamp = 0, box_result[3] = {0, 0, 0};  // the last stamp and counts
  uint32_t box_ghosts = 0;  // ghost bricks the pairs refresh
  bool box_affine = false;
  uint32_t box_base = 0, box_stride[3] = {0, 0, 0};
  uint32_t box_nb[3] = {0, 0, 0};
  uint32_t box_npairs = 0;
  bool march = false;  // the cube marches the units at every size
};

namespace {
std::atomic<uint64_t> g_next_plan_id{1};
}

namespace bk {

const PlanView plan_view(const bk_plan_s *p) {
  PlanView v;
  v.shape = p->shape;
  v.kcol = p->kcol;
  v.nunits = p->nunits;
  v.ncovered = p->ncovered;
  v.anchor = p->d_anchor;
  v.len = p->d_len;
  v.mask = p->d_mask;
  v.flat = p->d_flat;
  v.start = p->d_start;
  v.longest = p->longest;
  v.nbricks = p->nbricks;
  v.id = p->id;
  v.box_ids = p->d_box.load(std::memory_order_acquire);  // before what goes with it
  v.box_adj = p->d_box_adj;
  v.box_affine = p->box_affine;
  v.box_base = p->box_base;
  for (int a = 0; a < 3; ++a) {
    v.box_nb[a] = p->box_nb[a];
    v.box_stride[a] = p->box_stride[a];
  }
  v.box_npairs = p->box_npairs;
  v.march = p->march;
  return v;
}

void plan_march(bk_plan_s *p) { p->march = true; }

namespace {
// The device tables bound to the plans' boxes (bk_plan_bind_box): a sequence
// takes what the box stands for in place of its own tables only if they are
// among these, so what the library writes or frees in them ends the binding.
struct BoxTables {
  const uint32_t *adj, *pairs, *img_off, *img;  // pairs: null without ghost bricks
  std::array<std::pair<uintptr_t, uintptr_t>, 4> span;  // their bytes
};
constexpr size_t kMaxBound = 4;  // per plan; the oldest makes way
struct BoundTables {
  std::mutex mu;
  std::map<uint64_t, std::vector<BoxTables>> of;  // by plan id
  std::atomic<size_t> plans{0};                   // = of.size()
};
BoundTables &bound_tables() {
  static BoundTables *b = new BoundTables;  // frees at exit may still come
  return *b;
}
}  // namespace

bool box_bound(const PlanView &P, const uint32_t *adj, const uint32_t *pairs,
               const uint32_t *img_off, const uint32_t *img) {
  BoundTables &B = bound_tables();
  std::lock_guard<std::mutex> lock(B.mu);
  const auto it = B.of.find(P.id);
  if (it == B.of.end()) return false;
  for (const BoxTables &t : it->second)
    if (t.adj == adj && (!P.box_npairs || t.pairs == pairs) &&
        (!img_off || (t.img_off == img_off && t.img == img)))
      return true;
  return false;
}

void device_written(const void *p, size_t bytes) {
  BoundTables &B = bound_tables();
  if (!B.plans.load(std::memory_order_acquire)) return;
  const uintptr_t lo = reinterpret_cast<uintptr_t>(p), hi = lo + bytes;
  std::lock_guard<std::mutex> lock(B.mu);
  for (auto &entry : B.of) {
    auto &v = entry.second;
    v.erase(std::remove_if(v.begin(), v.end(),
                           [&](const BoxTables &t) {
                             return std::any_of(t.span.begin(), t.span.end(), [&](const auto &s) {
                               return s.first < hi && lo < s.second;
                             });
                           }),
            v.end());
  }
}

void device_freed(void *p) {
  if (!bound_tables().plans.load(std::memory_order_acquire)) return;
  hipDeviceptr_t base = p;
  size_t bytes = 1;
  if (hipMemGetAddressRange(&base, &bytes, p) != hipSuccess) {
    (void)hipGetLastError();
    base = p;
    bytes = 1;
  }
  device_written(base, bytes);
}

namespace {
void unbind_box(uint64_t plan) {
  BoundTables &B = bound_tables();
  std::lock_guard<std::mutex> lock(B.mu);
  B.of.erase(plan);
  B.plans.store(B.of.size(), std::memory_order_release);
}

// in place of older ones at the same addresses
void bind_box(uint64_t plan, const BoxTables &t) {
  BoundTables &B = bound_tables();
  std::lock_guard<std::mutex> lock(B.mu);
  auto &v = B.of[plan];
  B.plans.store(B.of.size(), std::memory_order_release);
  v.erase(std::remove_if(v.begin(), v.end(),
                         [&](const BoxTables &o) {
                           return o.adj == t.adj && o.pairs == t.pairs &&
                                  (!o.img_off || (o.img_off == t.img_off && o.img == t.img));
                         }),
          v.end());
  if (v.size() == kMaxBound) v.erase(v.begin());
  v.push_back(t);
}
}  // namespace

}  // namespace bk

namespace {

constexpr uint32_t kNone = UINT32_MAX;

// The units of a plan: unit u has its level-0 anchor and masks
// mask[first[u]] .. mask[first[u + 1] - 1], one per level.
struct Units {
  std::vector<uint32_t> anchor, first, mask;
  uint32_t count() const { return (uint32_t)anchor.size(); }
  uint32_t levels(uint32_t u) const { return first[u + 1] - first[u]; }
};

// Build k-chains of "cells" (a cell = one brick for columns, one quad level
// for quads) keyed by their anchor brick, then cut them into units.
void chain_cells(const uint32_t *adj, uint32_t nbricks, const std::vector<uint32_t> &cell_anchor,
                 const std::vector<uint32_t> &cell_mask, uint32_t kcol, Units &units) {
  std::vector<uint32_t> by_anchor(nbricks, kNone);  // an anchor's unused cell
  for (uint32_t c = 0; c < cell_anchor.size(); ++c) by_anchor[cell_anchor[c]] = c;
  units.first.push_back(0);
  units.mask.reserve(cell_anchor.size());
  for (uint32_t c = 0; c < cell_anchor.size(); ++c) {
    if (by_anchor[cell_anchor[c]] == kNone) continue;
    // walk up from c while the k+1 anchor is an unused cell
    uint32_t cur = c;
    uint32_t anchor = cell_anchor[cur];
    for (;;) {
      by_anchor[cell_anchor[cur]] = kNone;
      units.mask.push_back(cell_mask[cur]);
      if (units.mask.size() - units.first.back() == kcol) {
        units.anchor.push_back(anchor);
        units.first.push_back((uint32_t)units.mask.size());
      }
      const uint32_t up = adj[(size_t)cell_anchor[cur] * 27 + 22];
      if (by_anchor[up] == kNone) break;
      // the kernels hand a level's top planes to the next level as its k-1
      // face: link only where the adjacency agrees both ways (it does not
      // on the outer layer of a non-periodic grid, whose out-of-range
      // entries stand for no brick)
      if (adj[(size_t)up * 27 + 4] != cell_anchor[cur]) break;
      cur = by_anchor[up];
      if (units.mask.size() == units.first.back()) anchor = cell_anchor[cur];
    }
    if (units.mask.size() != units.first.back()) {
      units.anchor.push_back(anchor);
      units.first.push_back((uint32_t)units.mask.size());
    }
  }
}

// The quad kernel derives every input brick of a unit from its level-0
// anchor: members m1 = adj[m0][i+1], m2 = adj[m0][j+1], m3 = adj[m1][j+1];
// a 4x4 in-plane table of columns (entry (r, c) from m0 for r, c < 3, m1
// for column 3, m2 for row 3, m3 for the corner), level 0 from the members'
// in-plane neighbours, level -1 through adj[.][k-1], higher levels walked
// up through adj[.][k+1].  True when every stored member's 27 neighbours at
// every level are what those tables give -- always on a periodic grid and
// on the interior of a padded one, not on the outer layer of a
// non-periodic grid.
bool quad_unit_consistent(const uint32_t *adj, uint32_t anchor, const uint32_t *masks, int L,
                          std::vector<std::array<uint32_t, 16>> &T) {
  auto A = [adj](uint32_t b, int s) { return adj[(size_t)b * 27 + s]; };
  const uint32_t m0 = anchor, m1 = A(m0, 14), m2 = A(m0, 16), m3 = A(m1, 16);
  T.resize((size_t)L + 2);  // T[l + 1]: level l
  for (int e = 0; e < 16; ++e) {
    const int r = e >> 2, c = e & 3;
    const uint32_t m = r < 3 ? (c < 3 ? m0 : m1) : (c < 3 ? m2 : m3);
    const uint32_t n0 = A(m, 9 + 3 * (r < 3 ? r : 2) + (c < 3 ? c : 2));
    T[1][e] = n0;
    T[0][e] = A(n0, 4);
  }
  for (int l = 1; l <= L; ++l)
    for (int e = 0; e < 16; ++e) T[(size_t)l + 1][e] = A(T[l][e], 22);
  uint32_t om[4] = {m0, m1, m2, m3};
  for (int l = 0; l < L; ++l) {
    if (l > 0)
      for (auto &b : om) b = A(b, 22);
    for (int mm = 0; mm < 4; ++mm) {
      if (!((masks[l] >> mm) & 1u)) continue;
      for (int kd = 0; kd < 3; ++kd)
        for (int jd = 0; jd < 3; ++jd)
          for (int id = 0; id < 3; ++id)
            if (A(om[mm], kd * 9 + jd * 3 + id) !=
                T[(size_t)l + kd][((mm >> 1) + jd) * 4 + (mm & 1) + id])
              return false;
    }
  }
  return true;
}

}  // namespace

namespace {

// The wrapped box's brick next to its q-th in direction e.
__device__ __forceinline__ uint32_t wrapped(const uint32_t *__restrict__ ids, uint32_t nb0,
                                            uint32_t nb1, uint32_t nb2, uint32_t q, uint32_t e) {
  const uint32_t i = q % nb0, j = q / nb0 % nb1, k = q / nb0 / nb1;
  const uint32_t ii = (i + nb0 + e % 3 - 1) % nb0, jj = (j + nb1 + e / 3 % 3 - 1) % nb1,
                 kk = (k + nb2 + e / 9 - 1) % nb2;
  return ids[(kk * nb1 + jj) * nb0 + ii];
}

// adj[ids[q]][e] = wrapped(q, e), thread 27 q + e: neighbouring lanes, words
__global__ __launch_bounds__(256) void wrap_adjacency(const uint32_t *__restrict__ ids, uint32_t n,
                                                      uint32_t nb0, uint32_t nb1, uint32_t nb2,
                                                      uint32_t *__restrict__ adj) {
  const uint64_t t = (uint64_t)blockIdx.x * 256 + threadIdx.x;
  const uint32_t q = (uint32_t)(t / 27), e = (uint32_t)(t % 27);
  if (q < n) adj[(size_t)ids[q] * 27 + e] = wrapped(ids, nb0, nb1, nb2, q, e);
}

// Whether device tables are those of a declared box, by what each brick holds
// after a refresh (bk_plan_set_box): result[0] counts entries that are not,
// result[1] and result[2] the ghost bricks that the pairs and the images name,
// each once (stamped in seen).  The counts go on from check to check.
struct BoxCheck {
  const uint32_t *ids;    // [n]
  const uint32_t *holds;  // [nbricks]
  uint32_t *seen;         // [nbricks]
  uint32_t *result;
  const uint32_t *adj, *pairs, *off, *img;  // off, img: may be null
  uint32_t n, nbricks, nb0, nb1, nb2, npairs, stamp, bad;  // bad: result[0] before the check

  // ghost brick dst takes src's values: whether it is named for the first time
  __device__ __forceinline__ bool ghost(uint32_t dst, uint32_t src, uint32_t as, bool &bad) const {
    const bool is = dst < nbricks && dst != src && holds[dst] == src;
    bad = bad || !is;
    return is && atomicExch(&seen[dst], as) != as;
  }
};

// *count += x of all lanes (of one address: an atomic a wave, not a lane)
__device__ __forceinline__ void count_wave(uint32_t *count, uint32_t x) {
#pragma unroll
  for (int m = 1; m < 64; m <<= 1) x += __shfl_xor(x, m);
  if (x && (threadIdx.x & 63) == 0) atomicAdd(count, x);
}

// blockIdx.y 0, thread 27 q + e: neighbour e of the box's q-th brick; 1: pairs; 2:
// off rises from 0 to npairs, so that check_images stays in a table of as many.
__global__ __launch_bounds__(256) void check_tables(const BoxCheck c) {
  const uint64_t t = (uint64_t)blockIdx.x * 256 + threadIdx.x;
  bool bad = false;
  uint32_t named = 0;
  if (blockIdx.y == 0) {
    const uint32_t q = (uint32_t)(t / 27), e = (uint32_t)(t % 27);
    if (q < c.n) {
      const uint32_t b = c.adj[(size_t)c.ids[q] * 27 + e];
      bad = b >= c.nbricks || c.holds[b] != wrapped(c.ids, c.nb0, c.nb1, c.nb2, q, e);
    }
  } else if (blockIdx.y == 1) {
    if (t < c.npairs) named = c.ghost(c.pairs[2 * t], c.pairs[2 * t + 1], c.stamp, bad);
  } else if (t < c.nbricks) {
    bad = c.off[t] > c.off[t + 1] || (t == 0 && (c.off[0] != 0 || c.off[c.nbricks] != c.npairs));
  }
  count_wave(&c.result[0], bad);
  count_wave(&c.result[1], named);
}

__global__ __launch_bounds__(256) void check_images(const BoxCheck c) {
  if (__hip_atomic_load(&c.result[0], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != c.bad)
    return;  // (another block may have counted: as good a reason)
  const uint32_t q = blockIdx.x * 256 + threadIdx.x;
  bool bad = false;
  uint32_t named = 0;
  if (q < c.n) {
    const uint32_t b = c.ids[q];
    for (uint32_t t = c.off[b]; t < c.off[b + 1]; ++t)
      named += c.ghost(c.img[t], b, c.stamp + 1, bad);
  }
  count_wave(&c.result[0], bad);
  count_wave(&c.result[2], named);
}

// A plan's arrays on the host.
struct PlanArrays {
  std::vector<uint32_t> anchor, len, mask, flat, start;
};

int plan_build(const uint32_t *h_adj, uint32_t nbricks, const uint32_t *h_list, uint32_t nlist,
               int shape, uint32_t kcol, PlanArrays &out) {
  if (!h_adj || (nlist && !h_list))
    return bk::plan_fail(BK_ERR_ARG, "bk_plan_build_host: null pointer");
  if (shape != BK_PLAN_COLUMN && shape != BK_PLAN_QUAD)
    return bk::plan_fail(BK_ERR_ARG, "bk_plan: shape must be BK_PLAN_COLUMN or BK_PLAN_QUAD");
  if (kcol == 0 || kcol > 4096) return bk::plan_fail(BK_ERR_ARG, "bk_plan: kcol in [1, 4096]");
  for (uint32_t l = 0; l < nlist; ++l)
    if (h_list[l] >= nbricks) return bk::plan_fail(BK_ERR_ARG, "bk_plan: list entry out of range");
  uint32_t most = 0;
  for (size_t q = 0; q < (size_t)nbricks * 27; ++q) most = std::max(most, h_adj[q]);
  if (nbricks && most >= nbricks)
    return bk::plan_fail(BK_ERR_ARG, "bk_plan: adjacency entry out of range");

  // an entry's first position in the list (kNone: not listed)
  std::vector<uint32_t> pos(nbricks, kNone);
  for (uint32_t l = nlist; l-- > 0;) pos[h_list[l]] = l;
  std::vector<uint8_t> covered(nbricks, 0);

  std::vector<uint32_t> cell_anchor, cell_mask;
  for (uint32_t l = 0; l < nlist; ++l) {
    const uint32_t b = h_list[l];
    if (covered[b]) continue;
    if (shape == BK_PLAN_COLUMN) {
      covered[b] = 1;
      cell_anchor.push_back(b);
      cell_mask.push_back(1u);
    } else {
      const uint32_t m0 = b, m1 = h_adj[(size_t)m0 * 27 + 14], m2 = h_adj[(size_t)m0 * 27 + 16],
                     m3 = h_adj[(size_t)m1 * 27 + 16];
      const uint32_t mem[4] = {m0, m1, m2, m3};
      uint32_t mask = 0;
      for (int q = 0; q < 4; ++q) {
        bool dup = false;
        for (int p = 0; p < q; ++p) dup = dup || mem[p] == mem[q];
        if (!dup && pos[mem[q]] != kNone && !covered[mem[q]]) {
          covered[mem[q]] = 1;
          mask |= 1u << q;
        }
      }
      cell_anchor.push_back(m0);
      cell_mask.push_back(mask);
    }
  }
  Units units;
  chain_cells(h_adj, nbricks, cell_anchor, cell_mask, kcol, units);
  const uint32_t nu = units.count();
  if (shape == BK_PLAN_QUAD) {
    std::vector<std::array<uint32_t, 16>> tables;
    for (uint32_t u = 0; u < nu; ++u)
      if (!quad_unit_consistent(h_adj, units.anchor[u], &units.mask[units.first[u]],
                                (int)units.levels(u), tables))
        return bk::plan_fail(BK_ERR_UNSUPPORTED,
                             "bk_plan: a quad of the list has neighbours the adjacency does not "
                             "place consistently (the outer layer of a non-periodic grid); use "
                             "a column plan or no plan for such lists");
  }
  // emit units in the list order of their anchors (for a grid-ordered list:
  // k-segment by k-segment, so units that run together are neighbours)
  std::vector<std::pair<uint32_t, uint32_t>> key(nu);
  for (uint32_t u = 0; u < nu; ++u) key[u] = {pos[units.anchor[u]], u};
  std::stable_sort(key.begin(), key.end());

  out.anchor.resize(nu);
  out.len.resize(nu);
  out.start.resize(nu);
  out.mask.assign((size_t)nu * kcol, 0u);
  out.flat.clear();
  out.flat.reserve(nlist);
  for (uint32_t q = 0; q < nu; ++q) {
    const uint32_t u = key[q].second, L = units.levels(u);
    uint32_t a = units.anchor[u];
    out.start[q] = (uint32_t)out.flat.size();
    out.anchor[q] = a;
    out.len[q] = L;
    for (uint32_t l = 0; l < L; ++l) {
      const uint32_t m = units.mask[units.first[u] + l];
      out.mask[(size_t)q * kcol + l] = m;
      if (shape == BK_PLAN_COLUMN) {
        if (m & 1u) out.flat.push_back(a);
      } else {
        const uint32_t m1 = h_adj[(size_t)a * 27 + 14];
        const uint32_t mem[4] = {a, m1, h_adj[(size_t)a * 27 + 16], h_adj[(size_t)m1 * 27 + 16]};
        for (int b = 0; b < 4; ++b)
          if (m & (1u << b)) out.flat.push_back(mem[b]);
      }
      a = h_adj[(size_t)a * 27 + 22];
    }
  }
  return BK_OK;
}

}  // namespace

extern "C" {

int bk_plan_build_host(const uint32_t *h_adj, uint32_t nbricks, const uint32_t *h_list,
                       uint32_t nlist, int shape, uint32_t kcol, uint32_t *h_anchor,
                       uint32_t *h_len, uint32_t *h_mask, uint32_t *h_flat, uint32_t *nunits,
                       uint32_t *ncovered) {
  if (!nunits || !ncovered)
    return bk::plan_fail(BK_ERR_ARG, "bk_plan_build_host: null count pointer");
  PlanArrays A;
  const int rc = plan_build(h_adj, nbricks, h_list, nlist, shape, kcol, A);
  if (rc != BK_OK) return rc;
  auto put = [](uint32_t *dst, const std::vector<uint32_t> &v) {
    if (dst) std::copy(v.begin(), v.end(), dst);
  };
  put(h_anchor, A.anchor);
  put(h_len, A.len);
  put(h_mask, A.mask);
  put(h_flat, A.flat);
  *nunits = (uint32_t)A.anchor.size();
  *ncovered = (uint32_t)A.flat.size();
  return BK_OK;
}

}  // extern "C"

extern "C" {

int bk_plan_create(const uint32_t *h_adj, uint32_t nbricks, const uint32_t *h_list,
                   uint32_t nlist, int shape, uint32_t kcol, bk_plan *out) {
  if (!out) return bk::plan_fail(BK_ERR_ARG, "bk_plan_create: null out pointer");
  *out = nullptr;
  PlanArrays A;
  const int rc = plan_build(h_adj, nbricks, h_list, nlist, shape, kcol, A);
  if (rc != BK_OK) return rc;

  bk_plan_s *p = new bk_plan_s();
  p->shape = shape;
  p->kcol = kcol;
  p->nunits = (uint32_t)A.anchor.size();
  p->ncovered = (uint32_t)A.flat.size();
  for (uint32_t l : A.len) p->longest = std::max(p->longest, l);
  p->nbricks = nbricks;
  p->id = g_next_plan_id.fetch_add(1);
  (void)hipGetDevice(&p->device);  // the current device owns the arrays below
  // one allocation and one copy for all arrays, each from a 256-byte boundary
  const std::vector<uint32_t> *arr[5] = {&A.anchor, &A.len, &A.mask, &A.flat, &A.start};
  uint32_t **dst[5] = {&p->d_anchor, &p->d_len, &p->d_mask, &p->d_flat, &p->d_start};
  size_t at[5], total = 0;
  for (int q = 0; q < 5; ++q) {
    at[q] = total;
    total += (arr[q]->size() + 63) & ~(size_t)63;
  }
  if (total) {
    std::vector<uint32_t> all(total, 0u);
    for (int q = 0; q < 5; ++q)
      std::copy(arr[q]->begin(), arr[q]->end(), all.begin() + (ptrdiff_t)at[q]);
    hipError_t e = hipMalloc(&p->d_arrays, total * sizeof(uint32_t));
    if (e == hipSuccess)
      e = hipMemcpy(p->d_arrays, all.data(), total * sizeof(uint32_t), hipMemcpyHostToDevice);
    if (e != hipSuccess) {
      bk_plan_destroy(p);
      std::string m = std::string("bk_plan_create: ") + hipGetErrorString(e);
      return bk::plan_fail(e == hipErrorOutOfMemory ? BK_ERR_NOMEM : BK_ERR_HIP, m.c_str());
    }
    for (int q = 0; q < 5; ++q)
      if (!arr[q]->empty()) *dst[q] = p->d_arrays + at[q];
  }
  p->covered.assign(nbricks, false);
  for (uint32_t b : A.flat) p->covered[b] = true;
  *out = p;
  return BK_OK;
}

int bk_plan_destroy(bk_plan p) {
  if (!p) return BK_OK;
  // cached graphs captured the plan's device arrays: drop them first
  bk::graphs_forget_plan(p->id);
  bk::unbind_box(p->id);
  (void)hipFree(p->d_arrays);
  (void)hipFree(p->d_box.load());
  delete p;
  return BK_OK;
}

namespace {
// Allocations and copies of this thread while one of its streams is capturing:
// they are not part of the capture.
struct OutsideCapture {
  hipStreamCaptureMode mode = hipStreamCaptureModeRelaxed;
  OutsideCapture() { (void)hipThreadExchangeStreamCaptureMode(&mode); }
  ~OutsideCapture() { (void)hipThreadExchangeStreamCaptureMode(&mode); }
};

// The stream for them: the caller's, or while that is capturing one of our own
// per device, kept until the process ends (creating one takes 4 ms).
hipError_t setup_stream(hipStream_t &s) {
  hipStreamCaptureStatus capturing = hipStreamCaptureStatusNone;
  if (hipStreamIsCapturing(s, &capturing) != hipSuccess) (void)hipGetLastError();
  if (capturing == hipStreamCaptureStatusNone) return hipSuccess;
  static std::mutex mu;
  static std::map<int, hipStream_t> streams;
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return e;
  std::lock_guard<std::mutex> lock(mu);
  hipStream_t &kept = streams[dev];
  if (!kept) e = hipStreamCreateWithFlags(&kept, hipStreamNonBlocking);
  s = kept;
  return e;
}
}  // namespace

int bk_plan_set_box(bk_plan p, const uint32_t *h_adj, const long nb[3], const uint32_t *h_ids,
                    const uint32_t *h_pairs, uint32_t npairs, bk_stream stream) {
  if (!p || !h_adj || !nb || !h_ids || (npairs && !h_pairs))
    return bk::plan_fail(BK_ERR_ARG, "bk_plan_set_box: null pointer");
  std::lock_guard<std::mutex> lock(p->box_mu);
  if (p->d_box.load())
    return bk::plan_fail(BK_ERR_ARG, "bk_plan_set_box: the plan has a box already");
  for (int a = 0; a < 3; ++a)
    if (nb[a] <= 0 || nb[a] > (long)p->nbricks)
      return bk::plan_fail(BK_ERR_ARG, "bk_plan_set_box: bricks per axis out of range");
  const uint64_t plane = (uint64_t)nb[0] * (uint64_t)nb[1];
  if (plane > p->nbricks || plane * (uint64_t)nb[2] != p->ncovered)
    return bk::plan_fail(BK_ERR_UNSUPPORTED,
                         "bk_plan_set_box: the box does not have the plan's brick count");
  // what each brick holds before a sweep: itself, or for a ghost brick the
  // brick its pair copies onto it
  const size_t n = p->ncovered, nbr = p->nbricks, at = (n + 63) & ~(size_t)63;
  std::vector<uint32_t> upload;  // the ids, what each holds from `at`
  try {
    upload.assign(at + ((nbr + 63) & ~(size_t)63), kNone);
  } catch (const std::bad_alloc &) {
    return bk::plan_fail(BK_ERR_NOMEM, "bk_plan_set_box: out of host memory");
  }
  uint32_t *holds = upload.data() + at;
  std::copy(h_ids, h_ids + n, upload.begin());
  for (size_t q = 0; q < n; ++q) {
    const uint32_t b = h_ids[q];
    if (b >= p->nbricks || !p->covered[b] || holds[b] != kNone)
      return bk::plan_fail(BK_ERR_UNSUPPORTED,
                           "bk_plan_set_box: the box is not the plan's bricks, each once");
    holds[b] = b;
  }
  for (uint32_t q = 0; q < npairs; ++q) {
    const uint32_t dst = h_pairs[2 * q], src = h_pairs[2 * q + 1];
    if (dst >= p->nbricks || src >= p->nbricks || p->covered[dst])
      return bk::plan_fail(BK_ERR_UNSUPPORTED,
                           "bk_plan_set_box: a pair does not copy onto a ghost brick");
    holds[dst] = src;
  }
  // every neighbour of every box brick holds the brick the wrapped box has
  // there, so sweeps may read that brick instead
  size_t q = 0;
  for (long k = 0; k < nb[2]; ++k)
    for (long j = 0; j < nb[1]; ++j) {
      const uint32_t *row[9];
      for (int e = 0; e < 9; ++e) {
        const long kk = (k + e / 3 - 1 + nb[2]) % nb[2], jj = (j + e % 3 - 1 + nb[1]) % nb[1];
        row[e] = h_ids + ((size_t)kk * (size_t)nb[1] + (size_t)jj) * (size_t)nb[0];
      }
      for (long i = 0; i < nb[0]; ++i, ++q) {
        const uint32_t *ab = h_adj + (size_t)h_ids[q] * 27;
        const long at[3] = {i ? i - 1 : nb[0] - 1, i, i + 1 < nb[0] ? i + 1 : 0};
        for (int e = 0; e < 9; ++e)
          for (int d = 0; d < 3; ++d) {
            const uint32_t b = ab[e * 3 + d], want = row[e][at[d]];
            // (a box brick holds itself)
            if (b != want && (b >= p->nbricks || holds[b] != want))
              return bk::plan_fail(BK_ERR_UNSUPPORTED,
                                   "bk_plan_set_box: the adjacency and pairs are not those of a "
                                   "periodic box in this order");
          }
      }
    }
  // a box with ghost bricks gets an adjacency without them (a sequence that is
  // being captured may be the first over the plan)
  const OutsideCapture outside;
  // behind what is uploaded, cleared: the adjacency (ghost bricks' rows stay
  // so, unused), stamps and counts
  const size_t clear = upload.size(), nadj = npairs ? nbr * 27 : 0, nclear = nadj + nbr + 3;
  uint32_t *d = nullptr;
  hipStream_t own = static_cast<hipStream_t>(stream);
  hipError_t e = hipMalloc(&d, (clear + nclear) * sizeof(uint32_t));
  if (e == hipSuccess) e = setup_stream(own);
  if (e == hipSuccess)
    e = hipMemcpyAsync(d, upload.data(), clear * sizeof(uint32_t), hipMemcpyHostToDevice, own);
  if (e == hipSuccess) e = hipMemsetAsync(d + clear, 0, nclear * sizeof(uint32_t), own);
  if (e == hipSuccess && nadj) {
    hipLaunchKernelGGL(wrap_adjacency, dim3((uint32_t)((27 * n + 255) / 256)), dim3(256), 0, own, d,
                       (uint32_t)n, (uint32_t)nb[0], (uint32_t)nb[1], (uint32_t)nb[2], d + clear);
    e = hipGetLastError();
  }
  if (e == hipSuccess) e = hipStreamSynchronize(own);
  if (e != hipSuccess) {
    (void)hipFree(d);
    (void)hipGetLastError();  // the next launch is not to report it
    std::string m = std::string("bk_plan_set_box: ") + hipGetErrorString(e);
    return bk::plan_fail(e == hipErrorOutOfMemory ? BK_ERR_NOMEM : BK_ERR_HIP, m.c_str());
  }
  p->d_box_adj = nadj ? d + clear : nullptr;
  p->d_box_holds = d + at;
  p->d_box_seen = d + clear + nadj;
  p->box_ghosts = (uint32_t)(nbr - (size_t)std::count(holds, holds + nbr, kNone) - n);
  for (int a = 0; a < 3; ++a) p->box_nb[a] = (uint32_t)nb[a];
  p->box_npairs = npairs;
  // ids that follow a rule (init_grid's numbering): steps from the first brick
  const size_t step[3] = {1, (size_t)nb[0], (size_t)plane};
  p->box_base = h_ids[0];
  for (int a = 0; a < 3; ++a) p->box_stride[a] = nb[a] > 1 ? h_ids[step[a]] - h_ids[0] : 0;
  p->box_affine = true;
  q = 0;
  for (uint32_t k = 0; k < p->box_nb[2] && p->box_affine; ++k)
    for (uint32_t j = 0; j < p->box_nb[1] && p->box_affine; ++j) {
      const uint32_t row = p->box_base + j * p->box_stride[1] + k * p->box_stride[2];
      bool same = true;
      for (uint32_t i = 0; i < p->box_nb[0]; ++i) same &= h_ids[q++] == row + i * p->box_stride[0];
      p->box_affine = same;
    }
  p->d_box.store(d, std::memory_order_release);
  return BK_OK;
}

int bk_plan_bind_box(bk_plan p, const uint32_t *d_adj, const uint32_t *d_pairs,
                     uint32_t npairs, const uint32_t *d_img_off, const uint32_t *d_img,
                     bk_stream stream) {
  if (!p || !d_adj || (npairs && !d_pairs) || !d_img_off != !d_img)
    return bk::plan_fail(BK_ERR_ARG, "bk_plan_bind_box: null pointer");
  std::lock_guard<std::mutex> lock(p->box_mu);
  const uint32_t *ids = p->d_box.load();
  if (!ids) return bk::plan_fail(BK_ERR_ARG, "bk_plan_bind_box: the plan has no box");
  if (npairs != p->box_npairs)
    return bk::plan_fail(BK_ERR_UNSUPPORTED, "bk_plan_bind_box: not as many pairs as the box has");
  const OutsideCapture outside;
  hipStream_t own = static_cast<hipStream_t>(stream);
  hipError_t e = setup_stream(own);
  const uint32_t n = p->ncovered, nbricks = p->nbricks;
  BoxCheck c;
  c.ids = ids;
  c.holds = p->d_box_holds;
  c.seen = p->d_box_seen;
  c.result = p->d_box_seen + nbricks;
  c.adj = d_adj;
  c.pairs = npairs ? d_pairs : nullptr;
  c.off = d_img_off;
  c.img = d_img;
  c.n = n;
  c.nbricks = nbricks;
  c.nb0 = p->box_nb[0];
  c.nb1 = p->box_nb[1];
  c.nb2 = p->box_nb[2];
  c.npairs = npairs;
  c.stamp = p->box_stamp + 1;
  p->box_stamp += 2;
  c.bad = p->box_result[0];
  uint32_t result[3] = {0, 0, 0};
  if (e == hipSuccess) {
    const uint64_t most = std::max<uint64_t>(27ull * n, std::max(npairs, nbricks));
    hipLaunchKernelGGL(check_tables, dim3((uint32_t)((most + 255) / 256), d_img_off ? 3 : 2),
                       dim3(256), 0, own, c);
    if (d_img_off && npairs)
      hipLaunchKernelGGL(check_images, dim3((n + 255) / 256), dim3(256), 0, own, c);
    e = hipGetLastError();
  }
  if (e == hipSuccess)
    e = hipMemcpyAsync(result, c.result, sizeof result, hipMemcpyDeviceToHost, own);
  if (e == hipSuccess) e = hipStreamSynchronize(own);
  const uint32_t *was = p->box_result;
  const bool same = e == hipSuccess && result[0] == was[0] &&
                    result[1] - was[1] == p->box_ghosts &&
                    (!d_img_off || result[2] - was[2] == p->box_ghosts);
  if (e == hipSuccess) std::copy(result, result + 3, p->box_result);
  if (e != hipSuccess) {
    std::string m = std::string("bk_plan_bind_box: ") + hipGetErrorString(e);
    return bk::plan_fail(BK_ERR_HIP, m.c_str());
  }
  if (!same)
    return bk::plan_fail(BK_ERR_UNSUPPORTED,
                         "bk_plan_bind_box: the tables are not those of the plan's box");
  const auto span = [](const uint32_t *t, size_t words) {
    const uintptr_t lo = reinterpret_cast<uintptr_t>(t);
    return std::make_pair(lo, t ? lo + 4 * words : lo);
  };
  try {
    bk::bind_box(p->id, {d_adj, c.pairs, d_img_off, d_img,
                         {span(d_adj, (size_t)nbricks * 27), span(c.pairs, 2 * (size_t)npairs),
                          span(d_img_off, (size_t)nbricks + 1), span(d_img, npairs)}});
  } catch (const std::bad_alloc &) {
    return bk::plan_fail(BK_ERR_NOMEM, "bk_plan_bind_box: out of host memory");
  }
  return BK_OK;
}

int bk_plan_unbind_box(bk_plan p) {
  if (!p) return bk::plan_fail(BK_ERR_ARG, "bk_plan_unbind_box: null plan");
  bk::unbind_box(p->id);
  return BK_OK;
}

int bk_plan_query(bk_plan p, uint32_t *nunits, uint32_t *kcol, int *shape,
                  uint32_t *ncovered) {
  if (!p) return bk::plan_fail(BK_ERR_ARG, "bk_plan_query: null plan");
  if (nunits) *nunits = p->nunits;
  if (kcol) *kcol = p->kcol;
  if (shape) *shape = p->shape;
  if (ncovered) *ncovered = p->ncovered;
  return BK_OK;
}

int bk_plan_download(bk_plan p, uint32_t *h_anchor, uint32_t *h_len, uint32_t *h_mask,
                     uint32_t *h_flat) {
  if (!p) return bk::plan_fail(BK_ERR_ARG, "bk_plan_download: null plan");
  auto down = [](uint32_t *dst, const uint32_t *src, size_t n) -> hipError_t {
    if (!dst || !src || n == 0) return hipSuccess;
    return hipMemcpy(dst, src, n * sizeof(uint32_t), hipMemcpyDeviceToHost);
  };
  hipError_t e = down(h_anchor, p->d_anchor, p->nunits);
  if (e == hipSuccess) e = down(h_len, p->d_len, p->nunits);
  if (e == hipSuccess) e = down(h_mask, p->d_mask, (size_t)p->nunits * p->kcol);
  if (e == hipSuccess) e = down(h_flat, p->d_flat, p->ncovered);
  if (e != hipSuccess) return bk::plan_fail(BK_ERR_HIP, hipGetErrorString(e));
  return BK_OK;
}

}  // extern "C"
