// bk_aux.hip -- ghost refresh, fills, FP64 reductions and array<->brick
// conversion kernels for gfx950.
#include <algorithm>

#include "bk_device.h"
#include "bk_internal.h"

namespace bk {
namespace {

// ---------------------------------------------------------------------------
// Periodic ghost refresh: one wave per (dst, src) pair, whole-brick copy in
// 16-byte vectors.  Stands in for the one-rank periodic MPI exchange of
// weak/main.hip.cpp:249-269 (ghost bricks receive their periodic image).
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(256) void ghost_copy16(char *__restrict__ base,
                                                    uint64_t step_bytes,
                                                    uint32_t vec_per_brick,
                                                    const uint32_t *__restrict__ pairs,
                                                    uint32_t npairs) {
  const uint32_t p = blockIdx.x * 4u + (threadIdx.x >> 6);
  if (p >= npairs) return;
  const int lane = threadIdx.x & 63;
  const uint32_t dst = pairs[2 * p], src = pairs[2 * p + 1];
  const uint4 *s = reinterpret_cast<const uint4 *>(base + (size_t)src * step_bytes);
  uint4 *d = reinterpret_cast<uint4 *>(base + (size_t)dst * step_bytes);
  for (uint32_t v = lane; v < vec_per_brick; v += 64) d[v] = s[v];
}

// Whole-brick copy with NV 16-byte vectors per lane, every load issued
// before the first store (the generic loop above alternates them, since a
// store may alias the next load).
template <int NV>
__global__ __launch_bounds__(256) void ghost_copy16_n(char *__restrict__ base,
                                                      uint64_t step_bytes,
                                                      const uint32_t *__restrict__ pairs,
                                                      uint32_t npairs) {
  const uint32_t p = blockIdx.x * 4u + (threadIdx.x >> 6);
  if (p >= npairs) return;
  const int lane = threadIdx.x & 63;
  const uint32_t dst = pairs[2 * p], src = pairs[2 * p + 1];
  const uint4 *s = reinterpret_cast<const uint4 *>(base + (size_t)src * step_bytes);
  uint4 *d = reinterpret_cast<uint4 *>(base + (size_t)dst * step_bytes);
  uint4 t[NV];
#pragma unroll
  for (int q = 0; q < NV; ++q) t[q] = s[lane + 64 * q];
#pragma unroll
  for (int q = 0; q < NV; ++q) d[lane + 64 * q] = t[q];
}

__global__ __launch_bounds__(256) void ghost_copy2(char *__restrict__ base,
                                                   uint64_t step_bytes,
                                                   uint32_t half_per_brick,
                                                   const uint32_t *__restrict__ pairs,
                                                   uint32_t npairs) {
  const uint32_t p = blockIdx.x * 4u + (threadIdx.x >> 6);
  if (p >= npairs) return;
  const int lane = threadIdx.x & 63;
  const uint32_t dst = pairs[2 * p], src = pairs[2 * p + 1];
  const uint16_t *s = reinterpret_cast<const uint16_t *>(base + (size_t)src * step_bytes);
  uint16_t *d = reinterpret_cast<uint16_t *>(base + (size_t)dst * step_bytes);
  for (uint32_t v = lane; v < half_per_brick; v += 64) d[v] = s[v];
}

// ---------------------------------------------------------------------------
// streaming copy used to measure achievable HBM bandwidth: 16-byte vectors,
// four loads in flight per lane before their (non-temporal) stores
// ---------------------------------------------------------------------------
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));

__global__ __launch_bounds__(256) void stream_copy16(const u32x4 *__restrict__ s,
                                                     u32x4 *__restrict__ d, size_t n) {
  const size_t stride = (size_t)gridDim.x * 1024;
  size_t q = (size_t)blockIdx.x * 1024 + threadIdx.x;
  for (; q + 768 < n; q += stride) {
    const u32x4 t0 = s[q], t1 = s[q + 256], t2 = s[q + 512], t3 = s[q + 768];
    __builtin_nontemporal_store(t0, d + q);
    __builtin_nontemporal_store(t1, d + q + 256);
    __builtin_nontemporal_store(t2, d + q + 512);
    __builtin_nontemporal_store(t3, d + q + 768);
  }
  for (; q < n; q += 256) d[q] = s[q];
}

// ---------------------------------------------------------------------------
// register-only multiply-add loop used to measure the VALU rate the part
// sustains: C independent chains per lane, the coefficient wave-uniform (an
// SGPR operand, as in the stencil kernels), 64 FMAs per iteration
// ---------------------------------------------------------------------------
template <class T, int C>
__global__ __launch_bounds__(64) void valu_fma_probe(T *__restrict__ out, T c0, T c1,
                                                     uint32_t iters) {
  T acc[C], x[C];
#pragma unroll
  for (int i = 0; i < C; ++i) {
    acc[i] = T(threadIdx.x) * T(1e-3) + T(i);
    x[i] = T(threadIdx.x + i + 1) * T(0.5);
  }
  for (uint32_t it = 0; it < iters; ++it) {
#pragma unroll
    for (int r = 0; r < 32 / C; ++r)
#pragma unroll
      for (int i = 0; i < C; ++i) acc[i] = fmadd(c0, x[i], acc[i]);
#pragma unroll
    for (int r = 0; r < 32 / C; ++r)
#pragma unroll
      for (int i = 0; i < C; ++i) acc[i] = fmadd(c1, x[i], acc[i]);
  }
  T s = T(0);
#pragma unroll
  for (int i = 0; i < C; ++i) s += acc[i];
  out[(size_t)blockIdx.x * 64 + threadIdx.x] = s;
}

// Batched periodic refresh: one persistent launch refreshes the input field
// of every request of a table (all of one dtype); work item = one (dst,
// src) ghost pair of one request; NV 16-byte vectors per lane per brick.
template <int NV>
__global__ __launch_bounds__(256) void ghost_batched(const BatchTable *tab_, uint32_t tick) {
  const kconst_ptr<BatchTable> tab = (kconst_ptr<BatchTable>)tab_;
  const uint32_t nsegs = tab->nsegs;
  const uint32_t total = tab->prefix[nsegs];
  const uint32_t w = uniform(threadIdx.x >> 6);  // wave-uniform item, segment, pointers
  const int lane = threadIdx.x & 63;
  SegCursor cur;
  for (uint32_t p = blockIdx.x * 4u + w; p < total; p += gridDim.x * 4u) {
    cur.seek(tab->prefix, nsegs, p);
    const auto &sg = tab->seg[cur.s];
    if (tick >= sg.ticks) continue;
    const bool odd = ((sg.parity + tick) & 1u) != 0;
    char *base = static_cast<char *>(odd ? sg.f1 : sg.f0);
    const uint32_t q = p - cur.lo;
    const uint32_t dst = sg.items[2 * q], src = sg.items[2 * q + 1];
    const size_t step_bytes = (size_t)sg.step * (NV * 16 * 64 / 512);
    const uint4 *sp = reinterpret_cast<const uint4 *>(base + (size_t)src * step_bytes);
    uint4 *dp = reinterpret_cast<uint4 *>(base + (size_t)dst * step_bytes);
    uint4 t[NV];
#pragma unroll
    for (int v = 0; v < NV; ++v) t[v] = sp[lane + 64 * v];
#pragma unroll
    for (int v = 0; v < NV; ++v) dp[lane + 64 * v] = t[v];
  }
}

template <int NV>
hipError_t launch_ghost_batched_t(const BatchTable *tab, uint32_t tick, hipStream_t s) {
  static int nblk = 0;
  if (nblk == 0) {
    int dev = 0, cus = 256;
    (void)hipGetDevice(&dev);
    (void)hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev);
    nblk = cus * 8;
  }
  hipLaunchKernelGGL(ghost_batched<NV>, dim3(nblk), dim3(256), 0, s, tab, tick);
  return hipGetLastError();
}

// ---------------------------------------------------------------------------
// zero fill (a kernel, so it can sit inside a captured graph)
// ---------------------------------------------------------------------------
__global__ void zero16(uint4 *p, size_t n) {
  const size_t stride = (size_t)gridDim.x * blockDim.x;
  for (size_t q = (size_t)blockIdx.x * blockDim.x + threadIdx.x; q < n; q += stride)
    p[q] = make_uint4(0, 0, 0, 0);
}
__global__ void zero1(unsigned char *p, size_t n) {
  const size_t q = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (q < n) p[q] = 0;
}

// ---------------------------------------------------------------------------
// seeded uniform fill of the interior bricks (SplitMix64 finaliser of
// seed + (n+1)*golden, 53-bit uniform), same values as the oracle
// ---------------------------------------------------------------------------
// Brick extents (k, j, i) and vector fold (j, i) of a layout.
struct FoldGeom {
  uint32_t bk, bj, bi, fj, fi;
};

__device__ __forceinline__ uint64_t hash64(uint64_t seed, uint64_t n) {
  uint64_t z = seed + (n + 1) * 0x9E3779B97F4A7C15ULL;
  z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ULL;
  z = (z ^ (z >> 27)) * 0x94D049BB133111EBULL;
  return z ^ (z >> 31);
}

template <class T>
__global__ __launch_bounds__(256) void fill_uniform(T *__restrict__ dat, uint64_t step,
                                                    uint32_t nb0, uint32_t nb1,
                                                    uint32_t nb2, uint32_t ghost,
                                                    FoldGeom g, uint64_t seed, double lo,
                                                    double hi) {
  const uint64_t t = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const uint64_t nbricks = (uint64_t)nb0 * nb1 * nb2;
  if (t >= nbricks * 512) return;
  const uint64_t bi = t >> 9;
  const uint32_t e = (uint32_t)(t & 511);
  const uint32_t ti = (uint32_t)(bi % nb0), tj = (uint32_t)((bi / nb0) % nb1),
                 tk = (uint32_t)(bi / ((uint64_t)nb0 * nb1));
  // element e -> (k, j, i) through the fold: vector e / 64, lane e % 64
  const uint32_t vec = e >> 6, lane = e & 63;
  const uint32_t nj = g.bj / g.fj, ni = g.bi / g.fi;
  const uint32_t k = vec / (nj * ni);
  const uint32_t j = ((vec / ni) % nj) * g.fj + lane / g.fi;
  const uint32_t i = (vec % ni) * g.fi + lane % g.fi;
  const uint64_t n0 = (uint64_t)nb0 * g.bi, n1 = (uint64_t)nb1 * g.bj;
  const uint64_t x = (uint64_t)ti * g.bi + i, y = (uint64_t)tj * g.bj + j,
                 z = (uint64_t)tk * g.bk + k;
  const double u = (double)(hash64(seed, x + n0 * (y + n1 * z)) >> 11) * 0x1.0p-53;
  const double v = lo + (hi - lo) * u;
  const uint64_t S0 = nb0 + 2 * ghost, S1 = nb1 + 2 * ghost;
  const uint64_t b = (ti + ghost) + S0 * ((tj + ghost) + S1 * (tk + ghost));
  if constexpr (sizeof(T) == 8) {
    dat[b * step + e] = v;
  } else if constexpr (sizeof(T) == 4) {
    dat[b * step + e] = (float)v;
  } else {
    narrow(dat[b * step + e], (float)v);
  }
}

// ---------------------------------------------------------------------------
// FP64 reductions: every block reduces its share and writes one partial per
// value, the last block to finish combines the partials in block order
// (results do not depend on scheduling).  A thread takes C adjacent elements
// of four bricks at a time (16-byte loads where the element type allows, four
// in flight); the brick of a chunk is a shift away, not a division per
// element, and one ratio in compare's maximum needs its FP64 division only
// when it can be a new maximum of the wave.  Up to 256 blocks of 1024 threads: the
// last block starts from the count of blocks done, whose 1024 additions from
// smaller blocks took 7 us.  HBM bound: 256^3, us for the statistics of an
// FP32 field / the comparison of an FP32 with an FP64 one, 17.7 / 38 (3.8 and
// 5.3 TB/s) against 55 / 99 for one element a thread, a 64-bit division each
// and a second kernel.
// ---------------------------------------------------------------------------
constexpr int kReduceThreads = 1024;

template <class T> struct Elem;
template <> struct Elem<double> { typedef double type; };
template <> struct Elem<float> { typedef float type; };
template <> struct Elem<bf16> { typedef uint16_t type; };

__device__ __forceinline__ double to64(double x) { return x; }
__device__ __forceinline__ double to64(float x) { return (double)x; }
__device__ __forceinline__ double to64(uint16_t x) {
  return (double)__uint_as_float((uint32_t)x << 16);
}

// C adjacent elements at p (aligned as the element type)
template <class T, int C>
__device__ __forceinline__ void load64(const void *p, size_t at, double (&x)[C]) {
  typedef typename Elem<T>::type E;
  struct Chunk {
    E v[C];
  };
  const Chunk t = *reinterpret_cast<const Chunk *>(static_cast<const E *>(p) + at);
#pragma unroll
  for (int q = 0; q < C; ++q) x[q] = to64(t.v[q]);
}

// The largest value of the wave, NaN ignored, in every lane.
__device__ __forceinline__ double wave_max(double v) {
#pragma unroll
  for (int m = 1; m < 64; m <<= 1) v = fmax(v, __shfl_xor(v, m));
  return v;
}

// Sum (or maximum) of each value over the block's threads, in a fixed order,
// to thread 0.
template <int NV>
__device__ __forceinline__ void block_reduce(double (&v)[NV], const bool (&is_max)[NV],
                                             double (&sh)[NV][kReduceThreads / 64]) {
  auto across = [&](int q, int m) {
    const double o = __shfl_xor(v[q], m);
    v[q] = is_max[q] ? fmax(v[q], o) : v[q] + o;
  };
#pragma unroll
  for (int q = 0; q < NV; ++q) {
#pragma unroll
    for (int m = 1; m < 64; m <<= 1) across(q, m);
    if ((threadIdx.x & 63) == 0) sh[q][threadIdx.x >> 6] = v[q];
  }
  __syncthreads();
  if (threadIdx.x < 64) {
#pragma unroll
    for (int q = 0; q < NV; ++q) {
      v[q] = sh[q][threadIdx.x % (kReduceThreads / 64)];
#pragma unroll
      for (int m = 1; m < kReduceThreads / 64; m <<= 1) across(q, m);
    }
  }
  __syncthreads();
}

// A block's partials to part[block][NV]; the last block combines them all into
// out[0 .. NV).  *count rises by kReduceBlocks per launch, whatever its grid:
// by one a block and by what is left over with block 0, and the block that
// completes a multiple is the last.  Launches that overlap on one count spoil
// each other's results, but leave a multiple for those after them.
template <int NV>
__device__ __forceinline__ void finish(double (&v)[NV], const bool (&is_max)[NV], double *part,
                                       uint32_t *count, double *out) {
  __shared__ double sh[NV][kReduceThreads / 64];
  __shared__ bool last;
  block_reduce<NV>(v, is_max, sh);
  if (threadIdx.x == 0) {
#pragma unroll
    for (int q = 0; q < NV; ++q)
      __hip_atomic_store(&part[(size_t)blockIdx.x * NV + q], v[q], __ATOMIC_RELAXED,
                         __HIP_MEMORY_SCOPE_AGENT);
    // the partials, written through to memory every XCD reads, are there
    // before the count says so (a fence would write all of L2 back)
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    const uint32_t by = blockIdx.x ? 1u : kReduceBlocks + 1u - gridDim.x;
    last = (atomicAdd(count, by) + by) % kReduceBlocks == 0;
  }
  __syncthreads();
  if (!last) return;
#pragma unroll
  for (int q = 0; q < NV; ++q) v[q] = 0.0;
  for (uint32_t t = threadIdx.x; t < gridDim.x; t += kReduceThreads) {
#pragma unroll
    for (int q = 0; q < NV; ++q) {
      const double o = __hip_atomic_load(&part[(size_t)t * NV + q], __ATOMIC_RELAXED,
                                         __HIP_MEMORY_SCOPE_AGENT);
      v[q] = is_max[q] ? fmax(v[q], o) : v[q] + o;
    }
  }
  block_reduce<NV>(v, is_max, sh);
  if (threadIdx.x == 0) {
#pragma unroll
    for (int q = 0; q < NV; ++q) out[q] = v[q];
  }
}

// Calls body(bricks, chunks) for every chunk this thread owns of the listed
// bricks' `per` chunks each, U at a time (arrays of U, or of one at the end).
template <int U, class Body>
__device__ __forceinline__ void walk_chunks(const uint32_t *list, uint32_t nlist, uint32_t per,
                                            Body body) {
  if (per <= kReduceThreads && kReduceThreads % per == 0) {
    // several bricks a block at once, or one: no division in the loop
    const uint32_t bpb = kReduceThreads / per, sub = threadIdx.x / per, c = threadIdx.x - sub * per;
    const uint64_t stride = (uint64_t)gridDim.x * bpb;
    uint64_t l = (uint64_t)blockIdx.x * bpb + sub;
    for (; l + (U - 1) * stride < nlist; l += U * stride) {
      uint32_t b[U], e[U];
#pragma unroll
      for (int q = 0; q < U; ++q) {
        b[q] = list[l + q * stride];
        e[q] = c;
      }
      body(b, e);
    }
    for (; l < nlist; l += stride) {
      const uint32_t b[1] = {list[l]}, e[1] = {c};
      body(b, e);
    }
  } else {
    const uint64_t total = (uint64_t)nlist * per, stride = (uint64_t)gridDim.x * kReduceThreads;
    for (uint64_t t = (uint64_t)blockIdx.x * kReduceThreads + threadIdx.x; t < total; t += stride) {
      const uint64_t l = t / per;
      const uint32_t b[1] = {list[l]}, e[1] = {(uint32_t)(t - l * per)};
      body(b, e);
    }
  }
}

template <class T, int C>
__global__ __launch_bounds__(kReduceThreads) void stats_kernel(const void *dat, uint64_t step,
                                                    const uint32_t *list, uint32_t nlist,
                                                    uint32_t per, double *part, uint32_t *count,
                                                    double *out) {
  double s0[C] = {}, s1[C] = {}, s2[C] = {};
  walk_chunks<4>(list, nlist, per, [&](const auto &b, const auto &e) {
    constexpr int U = sizeof(b) / sizeof(b[0]);
    double x[U][C];
#pragma unroll
    for (int q = 0; q < U; ++q) load64<T, C>(dat, (size_t)b[q] * step + (size_t)e[q] * C, x[q]);
#pragma unroll
    for (int q = 0; q < U; ++q)
#pragma unroll
      for (int c = 0; c < C; ++c) {
        s0[c] += x[q][c];
        s1[c] += x[q][c] * x[q][c];
        s2[c] = fmax(s2[c], fabs(x[q][c]));
      }
  });
  double v[3] = {0.0, 0.0, 0.0};
#pragma unroll
  for (int c = 0; c < C; ++c) {
    v[0] += s0[c];
    v[1] += s1[c];
    v[2] = fmax(v[2], s2[c]);
  }
  const bool mx[3] = {false, false, true};
  finish<3>(v, mx, part, count, out);
}

template <class TA, class TR, int C>
__global__ __launch_bounds__(kReduceThreads) void compare_kernel(const void *a, uint64_t sa, const void *r,
                                                      uint64_t sr, const uint32_t *list,
                                                      uint32_t nlist, uint32_t per,
                                                      double floor_, double atol, double rtol,
                                                      double *part, uint32_t *count,
                                                      double *out) {
  double s0[C] = {}, s2[C] = {}, s3[C] = {};
  double ratio = 0.0, top = 0.0;  // this lane's largest ratio; a bound below the wave's
  uint64_t bad = 0;
  walk_chunks<2>(list, nlist, per, [&](const auto &b, const auto &e) {
    constexpr int U = sizeof(b) / sizeof(b[0]);
    double xa[U][C], xr[U][C];
#pragma unroll
    for (int q = 0; q < U; ++q) {
      load64<TA, C>(a, (size_t)b[q] * sa + (size_t)e[q] * C, xa[q]);
      load64<TR, C>(r, (size_t)b[q] * sr + (size_t)e[q] * C, xr[q]);
    }
    double d[U][C], den[U][C];
    bool more = false;
#pragma unroll
    for (int q = 0; q < U; ++q)
#pragma unroll
      for (int c = 0; c < C; ++c) {
        d[q][c] = fabs(xa[q][c] - xr[q][c]);
        const double m = fabs(xr[q][c]);
        den[q][c] = fmax(m, floor_);
        s0[c] = fmax(s0[c], d[q][c]);
        s2[c] += d[q][c] * d[q][c];
        s3[c] += xr[q][c] * xr[q][c];
        bad += (d[q][c] > atol + rtol * m) ? 1 : 0;
        // d / den can exceed top only where this holds (the product's
        // rounding is covered by the factor; a zero or underflowing product
        // holds too)
        more = more || d[q][c] >= top * den[q][c] * (1.0 - 0x1p-50);
      }
    if (__any(more)) {
#pragma unroll
      for (int q = 0; q < U; ++q)
#pragma unroll
        for (int c = 0; c < C; ++c) ratio = fmax(ratio, d[q][c] / den[q][c]);
      // lanes out of bricks would hand on anything: then each lane its own
      top = __ballot(1) == ~0ull ? wave_max(ratio) : ratio;
    }
  });
  double v[5] = {0.0, ratio, 0.0, 0.0, (double)bad};
#pragma unroll
  for (int c = 0; c < C; ++c) {
    v[0] = fmax(v[0], s0[c]);
    v[2] += s2[c];
    v[3] += s3[c];
  }
  const bool mx[5] = {true, true, false, false, false};
  finish<5>(v, mx, part, count, out);
}

// ---------------------------------------------------------------------------
// copyToBrick / copyFromBrick (bricksetup.h:139-221) on the device
// ---------------------------------------------------------------------------
struct CopyGeom {
  int64_t sa1, sa2;          // array strides (elements) for j and k
  int64_t pad0, pad1, pad2;  // padding per axis
  int64_t sb1, sb2;          // grid strides (bricks)
  int64_t k0, j0, i0;        // first brick per axis
  int64_t nk, nj, ni;        // bricks per axis in the iteration
};

// 16 bytes of cells, aligned as the element type (array rows start anywhere).
template <size_t ES> struct CellVec;
template <> struct CellVec<8> { typedef u32x4 type __attribute__((aligned(8))); };
template <> struct CellVec<4> { typedef u32x4 type __attribute__((aligned(4))); };
template <> struct CellVec<2> { typedef u32x4 type __attribute__((aligned(2))); };

// One wave moves R rows of B bricks side by side along i, 16 bytes a lane,
// for all eight planes (eight loads in flight): a load or store covers 128 to
// 512 contiguous bytes of every array row and 128 or 256 of every brick it
// touches.  HBM bound, at the copy rate.  One element a lane (a brick plane a
// wave: 64-byte pieces of eight array rows, half lines when storing to the
// array) against this, 400x264x312, us to bricks / back: FP64 142 / 152 ->
// 99 / 101 (rows off 16 bytes 144 / 168 -> 102 / 143), FP32 108 / 144 -> 51 /
// 53, BF16 103 / 102 -> 25 / 24.  R = 2 storing FP64 to the array: its rows
// may start anywhere, and longer runs leave fewer lines to two waves (off 16
// bytes 143 against 154 with R = 4; 8-byte-aligned otherwise equal).
constexpr int copy_rows(size_t es, bool to_brick) {
  return es == 2 ? 8 : es == 8 && !to_brick ? 2 : 4;
}

template <class T, bool TO_BRICK>
__global__ __launch_bounds__(256) void copy_brick(CopyGeom g, T *arr, const uint32_t *grid,
                                                  T *dat, uint64_t step) {
  typedef typename CellVec<sizeof(T)>::type Vec;
  constexpr int CPL = 16 / (int)sizeof(T), LPR = 8 / CPL;          // cells, lanes per row
  constexpr int R = copy_rows(sizeof(T), TO_BRICK), B = 64 / (LPR * R);  // rows, bricks of a wave
  constexpr int NRG = 8 / R;                                       // row groups of a brick
  const int lane = threadIdx.x & 63;
  const uint32_t w = blockIdx.x * 4u + uniform(threadIdx.x >> 6);
  const int64_t bi = (int64_t)(w / NRG) * B + (lane / LPR) % B;
  if (bi >= g.ni) return;
  const int row = (int)(w % NRG) * R + lane / (LPR * B), i = (lane % LPR) * CPL;
  const int64_t ti = g.i0 + bi;
  for (int64_t nk = blockIdx.z; nk < g.nk; nk += gridDim.z)
    for (int64_t nj = blockIdx.y; nj < g.nj; nj += gridDim.y) {
      const int64_t tj = g.j0 + nj, tk = g.k0 + nk;
      const size_t b = grid[ti + tj * g.sb1 + tk * g.sb2];
      T *pb = dat + b * step + row * 8 + i;
      T *pa = arr + ((g.pad0 + ti * 8 + i) + (g.pad1 + tj * 8 + row) * g.sa1 +
                     (g.pad2 + tk * 8) * g.sa2);
      Vec v[8];
#pragma unroll
      for (int k = 0; k < 8; ++k)
        v[k] = *reinterpret_cast<const Vec *>(TO_BRICK ? pa + k * g.sa2 : pb + k * 64);
#pragma unroll
      for (int k = 0; k < 8; ++k)
        *reinterpret_cast<Vec *>(TO_BRICK ? pb + k * 64 : pa + k * g.sa2) = v[k];
    }
}

template <class T>
hipError_t launch_copy_t(int to_brick, const CopyGeom &g, void *arr, const uint32_t *grid,
                         void *dat, size_t step, hipStream_t s) {
  if (g.nk <= 0 || g.nj <= 0 || g.ni <= 0) return hipSuccess;
  // waves along i: groups of 4 or 8 bricks, times the row groups (see the kernel)
  const int64_t R = copy_rows(sizeof(T), to_brick), B = 64 / (8 * (int64_t)sizeof(T) / 16 * R), NRG = 8 / R;
  const int64_t nx = ((g.ni + B - 1) / B * NRG + 3) / 4;
  const dim3 blocks((uint32_t)nx, (uint32_t)std::min<int64_t>(g.nj, 65535),
                    (uint32_t)std::min<int64_t>(g.nk, 65535));
  if (to_brick)
    hipLaunchKernelGGL((copy_brick<T, true>), blocks, dim3(256), 0, s, g, static_cast<T *>(arr),
                       grid, static_cast<T *>(dat), (uint64_t)step);
  else
    hipLaunchKernelGGL((copy_brick<T, false>), blocks, dim3(256), 0, s, g, static_cast<T *>(arr),
                       grid, static_cast<T *>(dat), (uint64_t)step);
  return hipGetLastError();
}

}  // namespace

hipError_t launch_ghost_refresh(void *dat, size_t step_bytes, size_t brick_bytes,
                                const uint32_t *pairs, uint32_t npairs, hipStream_t s) {
  if (npairs == 0) return hipSuccess;
  const uint32_t nwg = (npairs + 3u) / 4u;
  const bool v16 = (reinterpret_cast<uintptr_t>(dat) % 16 == 0) && (step_bytes % 16 == 0) &&
                   (brick_bytes % 16 == 0);
  char *b = static_cast<char *>(dat);
  if (v16 && brick_bytes == 4096)
    hipLaunchKernelGGL(ghost_copy16_n<4>, dim3(nwg), dim3(256), 0, s, b, (uint64_t)step_bytes,
                       pairs, npairs);
  else if (v16 && brick_bytes == 2048)
    hipLaunchKernelGGL(ghost_copy16_n<2>, dim3(nwg), dim3(256), 0, s, b, (uint64_t)step_bytes,
                       pairs, npairs);
  else if (v16 && brick_bytes == 1024)
    hipLaunchKernelGGL(ghost_copy16_n<1>, dim3(nwg), dim3(256), 0, s, b, (uint64_t)step_bytes,
                       pairs, npairs);
  else if (v16)
    hipLaunchKernelGGL(ghost_copy16, dim3(nwg), dim3(256), 0, s, b, (uint64_t)step_bytes,
                       (uint32_t)(brick_bytes / 16), pairs, npairs);
  else
    hipLaunchKernelGGL(ghost_copy2, dim3(nwg), dim3(256), 0, s, static_cast<char *>(dat),
                       (uint64_t)step_bytes, (uint32_t)(brick_bytes / 2), pairs, npairs);
  return hipGetLastError();
}

hipError_t launch_ghost_batched(int dtype, const BatchTable *tab, uint32_t tick, hipStream_t s) {
  switch (dtype) {
    case BK_F64: return launch_ghost_batched_t<4>(tab, tick, s);
    case BK_F32: return launch_ghost_batched_t<2>(tab, tick, s);
    case BK_BF16: return launch_ghost_batched_t<1>(tab, tick, s);
    default: return hipErrorInvalidValue;
  }
}

hipError_t launch_stream_copy(void *dst, const void *src, size_t bytes, hipStream_t s) {
  const size_t n = bytes / 16;
  if (n == 0) return hipSuccess;
  int dev = 0, cus = 256;
  (void)hipGetDevice(&dev);
  (void)hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev);
  size_t nblk = (n + 1023) / 1024;
  const size_t cap = (size_t)cus * 8;
  if (nblk > cap) nblk = cap;
  hipLaunchKernelGGL(stream_copy16, dim3((uint32_t)nblk), dim3(256), 0, s,
                     static_cast<const u32x4 *>(src), static_cast<u32x4 *>(dst), n);
  return hipGetLastError();
}

hipError_t launch_valu_probe(int dtype, int chains, uint32_t nblocks, uint32_t iters, void *out,
                             hipStream_t s) {
  const dim3 g(nblocks), b(64);
  if (dtype == BK_F64 && chains == 1)
    hipLaunchKernelGGL((valu_fma_probe<double, 1>), g, b, 0, s, static_cast<double *>(out),
                       0.999, 1.0001, iters);
  else if (dtype == BK_F64 && chains == 8)
    hipLaunchKernelGGL((valu_fma_probe<double, 8>), g, b, 0, s, static_cast<double *>(out),
                       0.999, 1.0001, iters);
  else if (dtype == BK_F32 && chains == 1)
    hipLaunchKernelGGL((valu_fma_probe<float, 1>), g, b, 0, s, static_cast<float *>(out),
                       0.999f, 1.0001f, iters);
  else if (dtype == BK_F32 && chains == 8)
    hipLaunchKernelGGL((valu_fma_probe<float, 8>), g, b, 0, s, static_cast<float *>(out),
                       0.999f, 1.0001f, iters);
  else
    return hipErrorInvalidValue;
  return hipGetLastError();
}

hipError_t launch_zero(void *dst, size_t bytes, hipStream_t s) {
  if (bytes == 0) return hipSuccess;
  unsigned char *p = static_cast<unsigned char *>(dst);
  size_t head = (16 - reinterpret_cast<uintptr_t>(p) % 16) % 16;
  if (head > bytes) head = bytes;
  if (head) hipLaunchKernelGGL(zero1, dim3(1), dim3(64), 0, s, p, head);
  const size_t nvec = (bytes - head) / 16;
  if (nvec) {
    size_t nblk = (nvec + 255) / 256;
    if (nblk > 65536) nblk = 65536;
    hipLaunchKernelGGL(zero16, dim3((uint32_t)nblk), dim3(256), 0, s,
                       reinterpret_cast<uint4 *>(p + head), nvec);
  }
  const size_t tail = bytes - head - nvec * 16;
  if (tail)
    hipLaunchKernelGGL(zero1, dim3(1), dim3(64), 0, s, p + head + nvec * 16, tail);
  return hipGetLastError();
}

hipError_t launch_fill_uniform(int layout, int dtype, void *dat, size_t step, const long nb[3],
                               int ghost, uint64_t seed, double lo, double hi, hipStream_t s) {
  const uint64_t n = (uint64_t)nb[0] * nb[1] * nb[2] * 512;
  if (n == 0) return hipSuccess;
  FoldGeom g;
  switch (layout) {
    case BK_LAYOUT_8x8x8: g = {8, 8, 8, 8, 8}; break;
    case BK_LAYOUT_4x8x16: g = {4, 8, 16, 4, 16}; break;
    case BK_LAYOUT_4x8x16_F88: g = {4, 8, 16, 8, 8}; break;
    default: return hipErrorInvalidValue;
  }
  const uint32_t nblk = (uint32_t)((n + 255) / 256);
  const uint32_t n0 = (uint32_t)nb[0], n1 = (uint32_t)nb[1], n2 = (uint32_t)nb[2];
  switch (dtype) {
    case BK_F64:
      hipLaunchKernelGGL(fill_uniform<double>, dim3(nblk), dim3(256), 0, s,
                         static_cast<double *>(dat), (uint64_t)step, n0, n1, n2,
                         (uint32_t)ghost, g, seed, lo, hi);
      break;
    case BK_F32:
      hipLaunchKernelGGL(fill_uniform<float>, dim3(nblk), dim3(256), 0, s,
                         static_cast<float *>(dat), (uint64_t)step, n0, n1, n2,
                         (uint32_t)ghost, g, seed, lo, hi);
      break;
    case BK_BF16:
      hipLaunchKernelGGL(fill_uniform<bf16>, dim3(nblk), dim3(256), 0, s,
                         static_cast<bf16 *>(dat), (uint64_t)step, n0, n1, n2,
                         (uint32_t)ghost, g, seed, lo, hi);
      break;
    default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

namespace {

// Blocks of a reduction over `chunks` chunks, U in flight a thread: no more than
// have work (the last block waits for a count of all of them).  100 bricks FP64,
// statistics / comparison, the kernel in us: 9.7 / 12.4 with 256 blocks, 8.2 /
// 11.3 with 7 and 13.
uint32_t reduce_blocks(uint64_t chunks, int U) {
  const uint64_t each = (uint64_t)kReduceThreads * U;
  return (uint32_t)std::min<uint64_t>(kReduceBlocks,
                                      std::max<uint64_t>(1, (chunks + each - 1) / each));
}

template <class T>
hipError_t launch_stats_t(const void *dat, size_t step, const uint32_t *list, uint32_t nlist,
                          size_t elems, double *part, uint32_t *count, double *out,
                          hipStream_t s) {
  constexpr int C = sizeof(T) == 8 ? 2 : sizeof(T) == 4 ? 4 : 8;  // 16 bytes
  const bool whole = elems % C == 0;
  const dim3 nb(reduce_blocks((uint64_t)nlist * elems / (whole ? C : 1), 4));
  if (whole)
    hipLaunchKernelGGL((stats_kernel<T, C>), nb, dim3(kReduceThreads), 0, s, dat,
                       (uint64_t)step, list, nlist, (uint32_t)(elems / C), part, count, out);
  else
    hipLaunchKernelGGL((stats_kernel<T, 1>), nb, dim3(kReduceThreads), 0, s, dat,
                       (uint64_t)step, list, nlist, (uint32_t)elems, part, count, out);
  return hipGetLastError();
}

template <class TA, class TR>
hipError_t launch_compare_t(const void *a, size_t sa, const void *r, size_t sr,
                            const uint32_t *list, uint32_t nlist, size_t elems, double floor_,
                            double atol, double rtol, double *part, uint32_t *count, double *out,
                            hipStream_t s) {
  // 16 bytes of the narrower type, at most four elements
  constexpr int C = sizeof(TA) == 8 && sizeof(TR) == 8 ? 2 : 4;
  const bool whole = elems % C == 0;
  const dim3 nb(reduce_blocks((uint64_t)nlist * elems / (whole ? C : 1), 2));
  if (whole)
    hipLaunchKernelGGL((compare_kernel<TA, TR, C>), nb, dim3(kReduceThreads), 0, s, a,
                       (uint64_t)sa, r, (uint64_t)sr, list, nlist, (uint32_t)(elems / C), floor_,
                       atol, rtol, part, count, out);
  else
    hipLaunchKernelGGL((compare_kernel<TA, TR, 1>), nb, dim3(kReduceThreads), 0, s, a,
                       (uint64_t)sa, r, (uint64_t)sr, list, nlist, (uint32_t)elems, floor_, atol,
                       rtol, part, count, out);
  return hipGetLastError();
}

template <class TA>
hipError_t launch_compare_a(int dtr, const void *a, size_t sa, const void *r, size_t sr,
                            const uint32_t *list, uint32_t nlist, size_t elems, double floor_,
                            double atol, double rtol, double *part, uint32_t *count, double *out,
                            hipStream_t s) {
  switch (dtr) {
    case BK_F64:
      return launch_compare_t<TA, double>(a, sa, r, sr, list, nlist, elems, floor_, atol, rtol,
                                          part, count, out, s);
    case BK_F32:
      return launch_compare_t<TA, float>(a, sa, r, sr, list, nlist, elems, floor_, atol, rtol,
                                         part, count, out, s);
    case BK_BF16:
      return launch_compare_t<TA, bf16>(a, sa, r, sr, list, nlist, elems, floor_, atol, rtol,
                                        part, count, out, s);
    default: return hipErrorInvalidValue;
  }
}

}  // namespace

hipError_t launch_field_stats(int dtype, const void *dat, size_t step, const uint32_t *list,
                              uint32_t nlist, size_t brick_elems, double *scratch,
                              uint32_t *count, double *out, hipStream_t s) {
  switch (dtype) {
    case BK_F64:
      return launch_stats_t<double>(dat, step, list, nlist, brick_elems, scratch, count, out, s);
    case BK_F32:
      return launch_stats_t<float>(dat, step, list, nlist, brick_elems, scratch, count, out, s);
    case BK_BF16:
      return launch_stats_t<bf16>(dat, step, list, nlist, brick_elems, scratch, count, out, s);
    default: return hipErrorInvalidValue;
  }
}

hipError_t launch_field_compare(int dta, const void *a, size_t step_a, int dtr, const void *r,
                                size_t step_r, const uint32_t *list, uint32_t nlist,
                                size_t brick_elems, double floor_, double atol, double rtol,
                                double *scratch, uint32_t *count, double *out, hipStream_t s) {
  switch (dta) {
    case BK_F64:
      return launch_compare_a<double>(dtr, a, step_a, r, step_r, list, nlist, brick_elems,
                                      floor_, atol, rtol, scratch, count, out, s);
    case BK_F32:
      return launch_compare_a<float>(dtr, a, step_a, r, step_r, list, nlist, brick_elems, floor_,
                                     atol, rtol, scratch, count, out, s);
    case BK_BF16:
      return launch_compare_a<bf16>(dtr, a, step_a, r, step_r, list, nlist, brick_elems, floor_,
                                    atol, rtol, scratch, count, out, s);
    default: return hipErrorInvalidValue;
  }
}

hipError_t launch_copy_brick(int to_brick, int dtype, const long dims[3], const long padding[3],
                             const long ghost[3], void *arr, const uint32_t *grid, void *dat,
                             size_t step, hipStream_t s) {
  CopyGeom g;
  const int64_t e0 = dims[0] + 2 * (padding[0] + ghost[0]);
  const int64_t e1 = dims[1] + 2 * (padding[1] + ghost[1]);
  g.sa1 = e0;
  g.sa2 = e0 * e1;
  g.pad0 = padding[0];
  g.pad1 = padding[1];
  g.pad2 = padding[2];
  const int64_t b0 = (dims[0] + 2 * ghost[0]) / 8, b1 = (dims[1] + 2 * ghost[1]) / 8;
  g.sb1 = b0;
  g.sb2 = b0 * b1;
  g.i0 = ghost[0] / 8;
  g.j0 = ghost[1] / 8;
  g.k0 = ghost[2] / 8;
  g.ni = (dims[0] + ghost[0]) / 8 - g.i0;
  g.nj = (dims[1] + ghost[1]) / 8 - g.j0;
  g.nk = (dims[2] + ghost[2]) / 8 - g.k0;
  switch (dtype) {
    case BK_F64: return launch_copy_t<double>(to_brick, g, arr, grid, dat, step, s);
    case BK_F32: return launch_copy_t<float>(to_brick, g, arr, grid, dat, step, s);
    case BK_BF16: return launch_copy_t<uint16_t>(to_brick, g, arr, grid, dat, step, s);
    default: return hipErrorInvalidValue;
  }
}

}  // namespace bk
