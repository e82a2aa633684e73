// bk_steps.hip -- several sweeps of a short-armed stencil (7- and 13-point star,
// cond) per pass over the field, for periodic boxes of 8x8x8 bricks on gfx950.
//
// bk_sweeps runs a loop of sweeps (weak/main.hip.cpp:274-279) whose every
// step reads and writes the whole field: past the caches' size each sweep
// costs a copy of the field, and a small box costs a launch per sweep.  Here
// one pass reads the field once, applies TS sweeps in registers and writes
// the result; the sweeps in between never reach memory.
//
// One wave owns a strip of J rows (j) of up to 7 bricks along i and marches
// along k.  Lane l holds one cell of every row.  The 64 cells of a row
// are the strip's and kHalo halo cells a side, laid round the wave as a ring --
// strip first, right halo, left halo -- so the i-taps are one-lane wave
// rotations (DPP) and groups of lanes fall on whole brick rows.  For each sweep
// s of the pass the wave keeps two planes of the field after s sweeps in
// registers (rows s .. NR-s-1 of the NR = J + 2 TS input rows).  When a new input plane arrives, each row goes through all TS
// sweeps at once:
//   n_{s+1}[r] = stencil of plane s around row r: centre row and rows r +- 1
//                from the newer kept plane, k+1 from n_s[r] just computed,
//                k-1 from the older kept plane,
// and n_s[r] then takes the older plane's place (the two planes swap roles
// from step to step).  Of sweep 0 the wave keeps the last loaded plane, the
// next one arriving while this one is used, and its older plane in LDS (each
// lane its own cells, so no barrier).  A sweep's halo (one row and one cell a
// side, one plane at either end of a march) is computed again by the
// neighbours instead of exchanged: no wave waits for another.
//
// Per point and sweep the arithmetic is the other star kernels': acc = c0*x,
// then fma over i+1, i-1, j+1, j-1, k+1, k-1; BF16 rounds after every sweep
// as a store would.  The bits are those of single sweeps.
//
// What bounds it (512^3, 7-point, TS = 4): the VALU and HBM about equally.
// FP64: 530 VALU instructions per wave and plane, 308 of them the stencil's;
// without any memory traffic the pass takes 0.40 ms, its 1.31 GB of reads and
// 1.07 GB of writes at the copy rate 0.45 ms; together 0.56 ms, 0.141 ms per
// sweep against 0.393 for one sweep per pass (FP32 0.086 against 0.203, BF16
// 0.089 against 0.117).  Three sweeps per pass: FP64 0.177, FP32 0.107 ms per
// sweep.  Found on the way: with the strip from the left halo on (lanes
// across brick edges) and one store per row 0.154; two cells a lane in FP32
// (fewer rotations, two waves per SIMD instead of three) no faster; issuing the
// first five taps of the next row among the last ones of this row, two rows
// per scheduling group, or loads two planes ahead no faster.
#include <algorithm>
#include <type_traits>

#include "bk_device.h"
#include "bk_internal.h"

namespace bk {
namespace {

constexpr int kHalo = 4;  // halo cells at either end of a row (TS <= 4)

// What the kernel computes: the 7-point star, or cond, keeping in registers
// the values themselves (taps clamp them at 0) or the clamped ones.  Clamped
// planes save the clamps of four taps in five; the select of the reference
// form needs no kept value, and with a threshold theta >= 0 a value exceeds
// theta exactly where its clamped one does.
enum Form { kStar = 0, kCondRaw = 1, kCondPos = 2, kStar13 = 3 };
constexpr int radius_of(int form) { return form == kStar13 ? 2 : 1; }

template <class T>
struct StepArgs {
  using A = typename acc_of<T>::type;
  const uint32_t *__restrict__ ids;  // box bricks, ids[(bk*nb1 + bj)*nb0 + bi]
  const T *__restrict__ in;
  T *__restrict__ out;
  uint64_t in_step;
  uint64_t out_step;
  uint32_t nb0, nb1, nb2;  // bricks of the box along i, j, k
  uint32_t affine, base, stride[3];  // affine: ids[...] = base + i, j, k by stride
  uint32_t nchunk;         // strips along i
  uint32_t njg;            // strips along j (nb1 * 8 / J)
  uint32_t njw;            // workgroups along j (four strips each)
  uint32_t ksegs;          // marches along k
  int cond_mode;
  A theta;
  A c[13];
};

// The value of the next (UP) or previous lane, the wave a ring of 64.
template <bool UP>
__device__ __forceinline__ uint32_t wave_turn32(uint32_t x) {
  return (uint32_t)__builtin_amdgcn_mov_dpp((int)x, UP ? 0x134 : 0x13c, 0xf, 0xf, true);
}
template <bool UP>
__device__ __forceinline__ float wave_turn(float x) {
  return __builtin_bit_cast(float, wave_turn32<UP>(__builtin_bit_cast(uint32_t, x)));
}
template <bool UP>
__device__ __forceinline__ double wave_turn(double x) {
  const uint64_t u = __builtin_bit_cast(uint64_t, x);
  const uint32_t lo = wave_turn32<UP>((uint32_t)u), hi = wave_turn32<UP>((uint32_t)(u >> 32));
  return __builtin_bit_cast(double, ((uint64_t)hi << 32) | lo);
}

// The value of the lane D above (UP) or below in its row of 16.
template <bool UP, int D>
__device__ __forceinline__ uint32_t row_next32(uint32_t x) {
  return (uint32_t)__builtin_amdgcn_mov_dpp((int)x, (UP ? 0x100 : 0x110) + D, 0xf, 0xf, true);
}
template <bool UP, int D>
__device__ __forceinline__ float row_next(float x) {
  return __builtin_bit_cast(float, row_next32<UP, D>(__builtin_bit_cast(uint32_t, x)));
}
template <bool UP, int D>
__device__ __forceinline__ double row_next(double x) {
  const uint64_t u = __builtin_bit_cast(uint64_t, x);
  const uint32_t lo = row_next32<UP, D>((uint32_t)u), hi = row_next32<UP, D>((uint32_t)(u >> 32));
  return __builtin_bit_cast(double, ((uint64_t)hi << 32) | lo);
}

// A cell of a plane.  (A struct: plain floats are allotted otherwise, and the
// sequences of 7-point sweeps took 1 % longer, FP32 360x216x264 471 -> 475 us,
// BF16 256^3 318 -> 322.)
template <class A>
struct Cell {
  A v;
};

// what a store to T and the next sweep's load make of a sweep's value
// (gfx950's conversion rounds as narrow() does: the same bits for all 2^32
// inputs)
template <class T, class A>
__device__ __forceinline__ A rounded(A x) {
  if constexpr (std::is_same<T, bf16>::value) {
    typedef float f2 __attribute__((ext_vector_type(2)));
    typedef __bf16 h2 __attribute__((ext_vector_type(2)));
    f2 t;
    t.x = t.y = x;
    return __uint_as_float(__builtin_bit_cast(uint32_t, __builtin_convertvector(t, h2)) << 16);
  }
  return x;
}

// Values of the lane `1` or `2` away in its group of four (quad_perm).
__device__ __forceinline__ uint32_t quad_swap1(uint32_t x) {
  return (uint32_t)__builtin_amdgcn_mov_dpp((int)x, 0xb1, 0xf, 0xf, true);
}
__device__ __forceinline__ uint32_t quad_swap2(uint32_t x) {
  return (uint32_t)__builtin_amdgcn_mov_dpp((int)x, 0x4e, 0xf, 0xf, true);
}
__device__ __forceinline__ double quad_swap1(double x) {
  const uint64_t u = __builtin_bit_cast(uint64_t, x);
  const uint32_t lo = quad_swap1((uint32_t)u), hi = quad_swap1((uint32_t)(u >> 32));
  return __builtin_bit_cast(double, ((uint64_t)hi << 32) | lo);
}

// Output rows in groups of G, each lane storing 16 bytes of one row of the
// group (a G x G exchange between G neighbouring lanes): a store instruction
// then covers 128 contiguous bytes per brick -- a whole line -- where one row
// is 64 (FP64) or 32 (FP32).  Row by row the FP64 pass took 0.62 ms against
// 0.58, the FP32 one 0.42 against 0.34.  BF16 keeps one store
// per row: an 8 x 8 exchange took it from 16.0 to 16.4 us a sweep at 256^3 (the
// VALU bounds it).
template <class T>
struct RowStore {
  static constexpr int G = 1;
  float x;
  __device__ __forceinline__ void put(int, float v) { x = v; }
  __device__ __forceinline__ void store(T *p, int, bool mine) const {
    if (mine) p->u = (uint16_t)(__float_as_uint(x) >> 16);  // already rounded to BF16
  }
};
template <>
struct RowStore<double> {
  static constexpr int G = 2;
  double x[2];
  __device__ __forceinline__ void put(int g, double v) { x[g] = v; }
  // p: the lane's cell in the group's first row
  __device__ __forceinline__ void store(double *p, int lane, bool mine) const {
    typedef double d2 __attribute__((ext_vector_type(2)));
    const bool odd = (lane & 1) != 0;
    const double got = quad_swap1(odd ? x[0] : x[1]);
    d2 v;
    v.x = odd ? got : x[0];
    v.y = odd ? x[1] : got;
    if (mine) *reinterpret_cast<d2 *>(p + (odd ? 7 : 0)) = v;
  }
};
template <>
struct RowStore<float> {
  static constexpr int G = 4;
  uint32_t x[4];
  __device__ __forceinline__ void put(int g, float v) { x[g] = __float_as_uint(v); }
  __device__ __forceinline__ void store(float *p, int lane, bool mine) const {
    typedef uint32_t u4 __attribute__((ext_vector_type(4)));
    const bool o1 = (lane & 1) != 0, o2 = (lane & 2) != 0;
    uint32_t y[4], z[4];
#pragma unroll
    for (int q = 0; q < 4; q += 2) {
      const uint32_t got = quad_swap1(o1 ? x[q] : x[q + 1]);
      y[q] = o1 ? got : x[q];
      y[q + 1] = o1 ? x[q + 1] : got;
    }
#pragma unroll
    for (int q = 0; q < 2; ++q) {
      const uint32_t got = quad_swap2(o2 ? y[q] : y[q + 2]);
      z[q] = o2 ? got : y[q];
      z[q + 2] = o2 ? y[q + 2] : got;
    }
    u4 v;
    v.x = z[0];
    v.y = z[1];
    v.z = z[2];
    v.w = z[3];
    if (mine) *reinterpret_cast<u4 *>(p + (lane & 3) * 7) = v;
  }
};

template <class T, int TS, int FORM>
__global__ __launch_bounds__(256)
__attribute__((amdgpu_waves_per_eu(2)))
void star_steps(const StepArgs<T> a) {
  using A = typename acc_of<T>::type;
  using X = Cell<A>;
  constexpr int J = 8, NR = J + 2 * TS;  // rows of the strip and of the input planes
  static_assert(TS >= 1 && TS <= kHalo, "the halo cells of a row");
  const int lane = threadIdx.x & 63;
  // each wave's older input plane, rows 1 .. NR-2, a lane its own cells
  __shared__ X older_all[4 * (NR - 2) * 64];
  X *older = older_all + (threadIdx.x >> 6) * ((NR - 2) * 64) + lane;

  // workgroup -> (march, four strips along j, strip along i)
  uint32_t w = xcd_remap(blockIdx.x, gridDim.x);
  const uint32_t ch = w % a.nchunk;
  w /= a.nchunk;
  const uint32_t jg = (w % a.njw) * 4u + uniform(threadIdx.x >> 6);
  const uint32_t seg = w / a.njw;
  if (jg >= a.njg) return;  // wave-uniform; nothing below synchronises waves

  // the strip along i: bricks [c0, c1); lane l cell l of it, the last
  // kHalo cells of the ring those before it (lanes past the right halo hold
  // further cells of the wrapped row, unused)
  const uint32_t c0 = a.nb0 * ch / a.nchunk, c1 = a.nb0 * (ch + 1) / a.nchunk;
  const uint32_t n0 = a.nb0 * 8, n1 = a.nb1 * 8, n2 = a.nb2 * 8;
  const int off = lane < 64 - kHalo ? lane : lane - 64;
  const uint32_t cell = (uint32_t)((int)(c0 * 8 + n0) + off) % n0;
  const uint32_t bi = cell >> 3, io = cell & 7;
  const bool mine = (uint32_t)lane < (c1 - c0) * 8;
  // rows: the strip's in brick row bj, the halo rows below and above in brick
  // rows bl and bh
  const uint32_t j0 = jg * J;
  const uint32_t jl = (j0 + n1 - 1) % n1, jh = (j0 + J) % n1;
  const uint32_t bj = j0 >> 3, bl = jl >> 3, bh = jh >> 3;
  // output planes [k0, k1)
  const uint32_t k0 = (uint32_t)((uint64_t)n2 * seg / a.ksegs),
                 k1 = (uint32_t)((uint64_t)n2 * (seg + 1) / a.ksegs);
  const int total = (int)(k1 - k0) + 2 * TS;

  // Input rows r - TS < 0 are read through pl, 0 .. J-1 through pc, J ..
  // through ph, at + (r - TS) * 8 (the pointers move 64 cells per plane).
  const int ol = ((int)(jl & 7) + 1) * 8 + (int)io, oc = (int)(j0 & 7) * 8 + (int)io,
            oh = ((int)(jh & 7) - J) * 8 + (int)io;
  auto id_of = [&](uint32_t lv, uint32_t b) { return a.ids[(lv * a.nb1 + b) * a.nb0 + bi]; };
  const uint32_t kf = (k0 + n2 - TS) % n2;  // first input plane (n2 >= 8 > TS)
  uint32_t lv = kf >> 3, kq = kf & 7;       // level, and the plane last loaded in it
  const T *pl, *pc, *ph;
  auto set_rows = [&](uint32_t il, uint32_t ic, uint32_t ih, int kofs) {
    pl = a.in + (size_t)il * a.in_step + (ol + kofs);
    pc = a.in + (size_t)ic * a.in_step + (oc + kofs);
    ph = a.in + (size_t)ih * a.in_step + (oh + kofs);
  };
  set_rows(id_of(lv, bl), id_of(lv, bj), id_of(lv, bh), (int)kq * 64);
  // brick ids one level ahead
  lv = lv + 1 == a.nb2 ? 0 : lv + 1;
  uint32_t nl = id_of(lv, bl), nc = id_of(lv, bj), nh = id_of(lv, bh);

  X ea[NR], eb[NR];  // the last input plane and the one arriving
  auto load_row = [&](int r, X(&e)[NR]) {
    const T *p = r < TS ? pl : (r < TS + J ? pc : ph);
    e[r].v = widen(p[(r - TS) * 8]);
  };
#pragma unroll
  for (int r = 0; r < NR; ++r) load_row(r, eb);

  uint32_t ko = k0;  // next output plane
  T *po = a.out + (size_t)id_of(k0 >> 3, bj) * a.out_step + ((int)(k0 & 7) * 64 + oc);

  X pa[TS][NR], pb[TS][NR];  // the two planes of sweeps 1 .. TS-1
#pragma unroll
  for (int r = 0; r < NR; ++r) {
    ea[r].v = A(0);
#pragma unroll
    for (int s = 0; s < TS; ++s) pa[s][r].v = pb[s][r].v = A(0);
  }

  // values as taps see them: of a kept plane, and of one just computed
  auto tap = [](A x) -> A {
    if constexpr (FORM == kCondRaw) return relu_ref(x);
    else return x;
  };
  auto keep = [](X x) -> X {
    if constexpr (FORM == kCondPos) x.v = relu_ref(x.v);
    return x;
  };
  // one sweep at one row: centre m, rows j+1 and j-1, planes k+1 and k-1
  auto point = [&](const X &m, const X &jp, const X &jm, const X &kp, const X &km) {
    const A t = tap(m.v);
    const A next = wave_turn<true>(t), prev = wave_turn<false>(t);
    A acc = a.c[0] * t;
    acc = fmadd(a.c[1], next, acc);
    acc = fmadd(a.c[2], prev, acc);
    acc = fmadd(a.c[3], tap(jp.v), acc);
    acc = fmadd(a.c[4], tap(jm.v), acc);
    acc = fmadd(a.c[5], tap(kp.v), acc);
    acc = fmadd(a.c[6], tap(km.v), acc);
    if constexpr (FORM != kStar) {
      const bool sel = a.cond_mode == 0 ? (acc > A(0)) : (m.v > a.theta);
      acc = sel ? acc : -acc;
    }
    return X{rounded<T>(acc)};
  };

  // One input plane F (E the one before it): every row through the TS sweeps.
  auto step = [&](X(&E)[NR], X(&F)[NR], X(&prv)[TS][NR], X(&cur)[TS][NR], int it) {
    // the next plane's addresses (past the last one needed, still a plane of
    // the box)
    if (++kq == 8) {
      kq = 0;
      set_rows(nl, nc, nh, 0);
      lv = lv + 1 == a.nb2 ? 0 : lv + 1;
      nl = id_of(lv, bl);
      nc = id_of(lv, bj);
      nh = id_of(lv, bh);
    } else {
      pl += 64;
      pc += 64;
      ph += 64;
    }
    const bool emit = it >= 2 * TS, st = emit && mine;
    // keeps the LDS plane in LDS (the compiler would carry it in registers)
    asm volatile("" ::: "memory");
    RowStore<T> rs;
    X km = older[0];
#pragma unroll
    for (int r = 0; r < NR; ++r) {
      X x = F[r] = keep(F[r]);
#pragma unroll
      for (int s = 0; s < TS; ++s) {
        if (r < s || r >= NR - s) continue;            // not a row of sweep s
        const bool in = r > s && r < NR - s - 1;       // sweep s+1 has the row too
        const int rm = r > 0 ? r - 1 : 0, rp = r + 1 < NR ? r + 1 : r;
        X o;
        if (s == 0) {
          if (in) {
            const X k0v = km;
            if (r + 2 < NR) km = older[r * 64];  // row r+1's
            o = point(E[r], E[rp], E[rm], x, k0v);
          }
          // row r-1 of E is done with: the older plane takes it, the next
          // plane's row comes in its place
          if (r > 1) older[(r - 2) * 64] = E[rm];
          if (r > 0) load_row(rm, E);
          if (r == NR - 1) load_row(r, E);
        } else {
          if (in) o = point(cur[s][r], cur[s][rp], cur[s][rm], x, prv[s][r]);
          prv[s][r] = x;
          // defined only here, after the older value's last use: the two can
          // share a register (the compiler's own copies sit at the loop's end
          // and doubled the registers held)
          if (in) asm volatile("" : "+v"(prv[s][r].v) : "v"(o.v));
        }
        if (in) x = s + 1 < TS ? keep(o) : o;
      }
      if (r >= TS && r < TS + J) {
        constexpr int G = RowStore<T>::G;
        const int q = r - TS;
        rs.put(q % G, x.v);
        if (q % G == G - 1) rs.store(po + (q - (G - 1)) * 8, lane, st);
      }
      __builtin_amdgcn_sched_barrier(0);  // row by row: bounds the live registers
    }
    if (emit) {
      ++ko;
      if ((ko & 7) == 0 && it + 1 < total)
        po = a.out + (size_t)id_of(ko >> 3, bj) * a.out_step + oc;
      else
        po += 64;
    }
  };
  for (int it = 0; it < total; it += 2) {
    step(ea, eb, pa, pb, it);
    if (it + 1 < total) step(eb, ea, pb, pa, it + 1);
  }
}

// The 13-point star (radius 2), two sweeps per pass: the same strips, halos and
// marches, so eight input planes for a first output.  A wave keeps in registers
// three planes of the input (the centre, the one above and the one arriving)
// and three of the field after one sweep; of both, what lies below the centre
// that still is needed is in LDS (two planes and one, each lane its own cells).
// The planes change roles from step to step, with a period of three.  Bound by
// memory and VALU about equally (210 registers in FP64: two waves per SIMD; 120
// in FP32).  us a sweep, one by one / so: FP64 256^3 60 / 39, 384^3 188 / 121,
// 512^3 434 / 289; FP32 256^3 36 / 27, 384^3 102 / 72, 512^3 228 / 167.  With E's
// rows loaded again wherever the scheduler liked, each row took two registers:
// 67 of FP64's spilled.
template <class T>
__global__ __launch_bounds__(256)
__attribute__((amdgpu_waves_per_eu(2)))
void star13_steps(const StepArgs<T> a) {
  using A = typename acc_of<T>::type;
  constexpr int R = 2, J = 8, H = 2 * R;
  constexpr int NR = J + 2 * H;   // rows of the input planes
  constexpr int N1 = J + 2 * R;   // rows after one sweep: R .. NR-R-1
  static_assert(H <= kHalo, "the halo cells of a row");
  const int lane = threadIdx.x & 63;
  __shared__ A older_all[4 * (2 * N1 + J) * 64];
  A *older = older_all + (threadIdx.x >> 6) * ((2 * N1 + J) * 64) + lane;
  A *older1 = older + 2 * N1 * 64;  // after one sweep, two planes below the centre
  int o1 = 0, o2 = N1 * 64;         // the input, one and two planes below

  // as in star_steps
  uint32_t w = xcd_remap(blockIdx.x, gridDim.x);
  const uint32_t ch = w % a.nchunk;
  w /= a.nchunk;
  const uint32_t jg = (w % a.njw) * 4u + uniform(threadIdx.x >> 6);
  const uint32_t seg = w / a.njw;
  if (jg >= a.njg) return;  // wave-uniform; nothing below synchronises waves
  const uint32_t c0 = a.nb0 * ch / a.nchunk, c1 = a.nb0 * (ch + 1) / a.nchunk;
  const uint32_t n0 = a.nb0 * 8, n1 = a.nb1 * 8, n2 = a.nb2 * 8;
  const int off = lane < 64 - kHalo ? lane : lane - 64;
  const uint32_t cell = (uint32_t)((int)(c0 * 8 + n0) + off) % n0;
  const uint32_t bi = cell >> 3, io = cell & 7;
  const bool mine = (uint32_t)lane < (c1 - c0) * 8;
  const uint32_t j0 = jg * J;
  const uint32_t jl = (j0 + n1 - 1) % n1, jh = (j0 + J) % n1;
  const uint32_t bj = j0 >> 3, bl = jl >> 3, bh = jh >> 3;
  const uint32_t k0 = (uint32_t)((uint64_t)n2 * seg / a.ksegs),
                 k1 = (uint32_t)((uint64_t)n2 * (seg + 1) / a.ksegs);
  const int total = (int)(k1 - k0) + 2 * H;
  const int ol = ((int)(jl & 7) + 1) * 8 + (int)io, oc = (int)(j0 & 7) * 8 + (int)io,
            oh = ((int)(jh & 7) - J) * 8 + (int)io;
  auto id_of = [&](uint32_t lv, uint32_t b) { return a.ids[(lv * a.nb1 + b) * a.nb0 + bi]; };
  const uint32_t kf = (k0 + n2 - H) % n2;
  uint32_t lv = kf >> 3, kq = kf & 7;
  const T *pl, *pc, *ph;
  auto set_rows = [&](uint32_t il, uint32_t ic, uint32_t ih, int kofs) {
    pl = a.in + (size_t)il * a.in_step + (ol + kofs);
    pc = a.in + (size_t)ic * a.in_step + (oc + kofs);
    ph = a.in + (size_t)ih * a.in_step + (oh + kofs);
  };
  set_rows(id_of(lv, bl), id_of(lv, bj), id_of(lv, bh), (int)kq * 64);
  lv = lv + 1 == a.nb2 ? 0 : lv + 1;
  uint32_t nl = id_of(lv, bl), nc = id_of(lv, bj), nh = id_of(lv, bh);

  A e0[NR], e1[NR], e2[NR];  // planes of the input
  A m0[NR], m1[NR], m2[NR];  // planes of the field after one sweep
  auto load_row = [&](int r, A(&e)[NR]) {
    const T *p = r < H ? pl : (r < H + J ? pc : ph);
    e[r] = widen(p[(r - H) * 8]);
  };
#pragma unroll
  for (int r = 0; r < NR; ++r) {
    e0[r] = e1[r] = m0[r] = m1[r] = m2[r] = A(0);
    load_row(r, e2);
  }
  uint32_t ko = k0;  // next output plane
  T *po = a.out + (size_t)id_of(k0 >> 3, bj) * a.out_step + ((int)(k0 & 7) * 64 + oc);

  // one sweep at row r of plane e; planes k + 1, k + 2, k - 1, k - 2
  auto point = [&](const A(&e)[NR], int r, A kp1, A kp2, A km1, A km2) {
    const A t = e[r];
    const A n1 = wave_turn<true>(t), p1 = wave_turn<false>(t);
    A acc = a.c[0] * t;
    acc = fmadd(a.c[1], n1, acc);
    acc = fmadd(a.c[2], p1, acc);
    acc = fmadd(a.c[3], e[r + 1], acc);
    acc = fmadd(a.c[4], e[r - 1], acc);
    acc = fmadd(a.c[5], kp1, acc);
    acc = fmadd(a.c[6], km1, acc);
    acc = fmadd(a.c[7], wave_turn<true>(n1), acc);
    acc = fmadd(a.c[8], wave_turn<false>(p1), acc);
    acc = fmadd(a.c[9], e[r + 2], acc);
    acc = fmadd(a.c[10], e[r - 2], acc);
    acc = fmadd(a.c[11], kp2, acc);
    return fmadd(a.c[12], km2, acc);
  };
  // one input plane F arrived, P the one before it, E the centre of the first
  // sweep; of the second, p the plane above the centre c and m the one below
  auto step = [&](A(&E)[NR], A(&P)[NR], A(&F)[NR], A(&c)[NR], A(&p)[NR], A(&m)[NR], int it) {
    if (++kq == 8) {
      kq = 0;
      set_rows(nl, nc, nh, 0);
      lv = lv + 1 == a.nb2 ? 0 : lv + 1;
      nl = id_of(lv, bl);
      nc = id_of(lv, bj);
      nh = id_of(lv, bh);
    } else {
      pl += 64;
      pc += 64;
      ph += 64;
    }
    const bool emit = it >= 2 * H, st = emit && mine;
    asm volatile("" ::: "memory");  // keeps the LDS planes in LDS
    RowStore<T> rs;
    A km1 = older[o1], km2 = older[o2], kn2 = older1[0];
    // row q of E is done with: it takes the place of the plane two below, the
    // next plane's row comes in its place
    auto release = [&](int q) {
      if (q >= R && q < NR - R) older[o2 + (q - R) * 64] = E[q];
      load_row(q, E);
    };
#pragma unroll
    for (int r = 0; r < NR; ++r) {
      if (r >= R && r < NR - R) {
        const A a1 = km1, a2 = km2;
        if (r + 1 < NR - R) {
          km1 = older[o1 + (r + 1 - R) * 64];
          km2 = older[o2 + (r + 1 - R) * 64];
        }
        A x = point(E, r, P[r], F[r], a1, a2);
        // loaded again only after x: the old and the new row share a register
        asm volatile("" : "+v"(E[r - R]) : "v"(x));
        release(r - R);
        if (r >= H && r < NR - H) {
          const A b2 = kn2;
          if (r + 1 < NR - H) kn2 = older1[(r + 1 - H) * 64];
          A y = point(c, r, p[r], x, m[r], b2);
          older1[(r - H) * 64] = m[r];
          constexpr int G = RowStore<T>::G;
          const int q = r - H;
          rs.put(q % G, y);
          m[r] = x;
          asm volatile("" : "+v"(m[r]) : "v"(y));
          if (q % G == G - 1) rs.store(po + (q - (G - 1)) * 8, lane, st);
        } else {
          m[r] = x;
        }
      } else if (r >= NR - R) {
        release(r - R);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    release(NR - 2);
    release(NR - 1);
    const int o = o1;
    o1 = o2;
    o2 = o;
    if (emit) {
      ++ko;
      if ((ko & 7) == 0 && it + 1 < total)
        po = a.out + (size_t)id_of(ko >> 3, bj) * a.out_step + oc;
      else
        po += 64;
    }
  };
  for (int it = 0;; it += 3) {
    step(e0, e1, e2, m0, m1, m2, it);
    if (it + 1 >= total) break;
    step(e1, e2, e0, m1, m2, m0, it + 1);
    if (it + 2 >= total) break;
    step(e2, e0, e1, m2, m0, m1, it + 2);
    if (it + 3 >= total) break;
  }
}

// Small boxes: one workgroup per brick (BK = 8) or half brick (BK = 4 planes)
// and pass, so that a few hundred bricks reach every CU.  The workgroup's 256
// threads are the 16 x 16 columns of the brick's plane and its 4 halo cells a
// side; a thread keeps its column's BK + 2 TS planes in registers.  Per sweep
// the columns' values go to LDS, the j-taps come from there, the i-taps by DPP
// from the 16-lane row (one row of the region), the k-taps from the thread's
// own registers; two LDS buffers in turn, so one barrier per sweep.
template <class T, int TS, int BK, int FORM>
__global__ __launch_bounds__(256) void star_steps_block(const StepArgs<T> a) {
  using A = typename acc_of<T>::type;
  constexpr int R = radius_of(FORM), H = TS * R;  // radius, halo planes a side
  constexpr int NP = BK + 2 * H;                  // planes of the input
  static_assert(TS >= 1 && H <= kHalo && H <= BK && (BK == 4 || BK == 8),
                "the halo planes of a side lie in one level");
  // buffer s & 1 of sweep s + 1: planes (s+1) R .. NP-(s+1)R-1 of the field
  // after s sweeps, from plane R (even s) or 2 R (odd s)
  __shared__ A lds[((NP - 2 * R) + (NP - 4 * R)) * 256];
  const int t = threadIdx.x, x = t & 15, y = t >> 4;
  uint32_t w = xcd_remap(blockIdx.x, gridDim.x);
  const uint32_t bi = w % a.nb0;
  w /= a.nb0;
  const uint32_t bj = w % a.nb1;
  const uint32_t k0 = w / a.nb1 * BK;  // first output plane
  const uint32_t n0 = a.nb0 * 8, n1 = a.nb1 * 8, n2 = a.nb2 * 8;
  // (kHalo before the box to kHalo + 7 past it: at most one box away)
  auto wrap = [](uint32_t v, uint32_t n) { return v < n ? v : (int)v < 0 ? v + n : v - n; };
  const uint32_t ci = wrap(bi * 8 - kHalo + x, n0), cj = wrap(bj * 8 - kHalo + y, n1);
  const uint32_t kl = k0 ? k0 - 1 : n2 - 1, kh = k0 + BK < n2 ? k0 + BK : 0;  // planes next to the block
  // computed where the ids follow a rule: the table is a load ahead of the loads
  uint32_t il, ic, ih;
  if (a.affine) {
    const uint32_t row = a.base + (cj >> 3) * a.stride[1] + (ci >> 3) * a.stride[0];
    il = row + (kl >> 3) * a.stride[2];
    ic = row + (k0 >> 3) * a.stride[2];
    ih = row + (kh >> 3) * a.stride[2];
  } else {
    const uint32_t row = (cj >> 3) * a.nb0 + (ci >> 3), per = a.nb0 * a.nb1;
    il = a.ids[(kl >> 3) * per + row];
    ic = a.ids[(k0 >> 3) * per + row];
    ih = a.ids[(kh >> 3) * per + row];
  }
  const int e = (int)((cj & 7) * 8 + (ci & 7));
  const T *pl = a.in + (size_t)il * a.in_step + (e + ((int)(kl & 7) + 1) * 64);
  const T *pc = a.in + (size_t)ic * a.in_step + (e + (int)(k0 & 7) * 64);
  const T *ph = a.in + (size_t)ih * a.in_step + (e + ((int)(kh & 7) - BK) * 64);
  A c[NP];
#pragma unroll
  for (int p = 0; p < NP; ++p) {
    const T *q = p < H ? pl : (p < H + BK ? pc : ph);
    c[p] = widen(q[(p - H) * 64]);
  }
  constexpr bool kCond = FORM == kCondRaw || FORM == kCondPos;
  auto tap = [](A v) -> A {
    if constexpr (kCond) return relu_ref(v);
    else return v;
  };
  int yp[R], ym[R];  // the columns at j + 1 .. j + R and j - 1 .. (of halo rows: any)
#pragma unroll
  for (int r = 0; r < R; ++r) {
    yp[r] = y + r < 15 ? t + (r + 1) * 16 : t;
    ym[r] = y > r ? t - (r + 1) * 16 : t;
  }
#pragma unroll
  for (int s = 0; s < TS; ++s) {
    A *buf = lds + (s & 1 ? (NP - 2 * R) * 256 : 0);
    const int p0 = ((s & 1) + 1) * R, lo = (s + 1) * R, hi = NP - (s + 1) * R;
#pragma unroll
    for (int p = lo; p < hi; ++p) buf[(p - p0) * 256 + t] = tap(c[p]);
    __syncthreads();
    A below[R];  // planes p - 1 .. p - R before this sweep
#pragma unroll
    for (int r = 0; r < R; ++r) below[r] = tap(c[lo - 1 - r]);
#pragma unroll
    for (int p = lo; p < hi; ++p) {
      const A m = tap(c[p]);
      const A *row = buf + (p - p0) * 256;
      A acc = a.c[0] * m;
      acc = fmadd(a.c[1], row_next<true, 1>(m), acc);
      acc = fmadd(a.c[2], row_next<false, 1>(m), acc);
      acc = fmadd(a.c[3], row[yp[0]], acc);
      acc = fmadd(a.c[4], row[ym[0]], acc);
      acc = fmadd(a.c[5], tap(c[p + 1]), acc);
      acc = fmadd(a.c[6], below[0], acc);
      if constexpr (R == 2) {
        acc = fmadd(a.c[7], row_next<true, 2>(m), acc);
        acc = fmadd(a.c[8], row_next<false, 2>(m), acc);
        acc = fmadd(a.c[9], row[yp[R - 1]], acc);
        acc = fmadd(a.c[10], row[ym[R - 1]], acc);
        acc = fmadd(a.c[11], c[p + R], acc);
        acc = fmadd(a.c[12], below[R - 1], acc);
      }
      if constexpr (kCond) {
        const bool sel = a.cond_mode == 0 ? (acc > A(0)) : (c[p] > a.theta);
        acc = sel ? acc : -acc;
      }
      if constexpr (R == 2) below[R - 1] = below[0];
      below[0] = m;
      c[p] = rounded<T>(acc);
    }
  }
  if (x >= kHalo && x < kHalo + 8 && y >= kHalo && y < kHalo + 8) {
    T *po = a.out + (size_t)ic * a.out_step + (e + (int)(k0 & 7) * 64);
#pragma unroll
    for (int p = H; p < H + BK; ++p) narrow(po[(p - H) * 64], c[p]);
  }
}

template <class T, int TS, int FORM>
auto strip_kernel() {
  if constexpr (FORM == kStar13) return &star13_steps<T>;
  else return &star_steps<T, TS, FORM>;
}

// How a box is cut into strips of 8 rows and marches along k.  Two workgroups
// (of four strips) per CU; more, shorter marches fill the device better and
// compute more halo planes.  us a sweep with one, two, three, four workgroups
// per CU: 7-point FP64 192^3 12.7, 12.5, 14.2, 16.0, FP32 10.6, 10.0, 10.6,
// 12.2, BF16 256^3 21.0, 17.4, 17.5, 19.1, 13-point FP32 192^3 19.3, 17.9, 18.6,
// 20.7.  In large boxes marches of at most 64 planes for four sweeps (512^3
// FP32 97.8 with 171, 93.9 with 64), 171 for fewer sweeps, which are bound by
// memory (three sweeps 107 against 117, 13-point FP32 167 against 181).
struct Strips {
  uint32_t nchunk, njg, njw, ksegs;
  Strips(const PlanView &P, int ts) {
    const uint32_t most = (64 - 2 * kHalo) / 8;  // bricks of a strip along i
    nchunk = (P.box_nb[0] + most - 1) / most;
    njg = P.box_nb[1];
    njw = (njg + 3) / 4;
    const uint64_t per = (uint64_t)nchunk * njw;  // workgroups of a march
    const uint32_t least = ts == 4 ? P.box_nb[2] / 8 : P.box_nb[2] / 21;
    uint64_t segs = std::min<uint64_t>(std::max<uint64_t>(512 / per, least), P.box_nb[2]);
    segs = std::max<uint64_t>(segs, 1);
    // a little more than the device takes at once (FP64) would wait for a
    // second turn of a few
    if (per * segs > 512 && per * segs < 768 && per <= 512) segs = 512 / per;
    // one a CU where the second would add less than it costs (18^3 bricks: 270
    // workgroups of 16 planes, a few CUs with two, against 255 of 17)
    const uint64_t one = 256 / per, n2 = (uint64_t)P.box_nb[2] * 8;
    if (one >= std::max<uint32_t>(least, 1) && one < segs &&
        2 * (n2 / one + 2 * kHalo) <= 3 * (n2 / segs + 2 * kHalo))
      segs = one;
    ksegs = (uint32_t)segs;
  }
  // of workgroups per CU: the fullest CU's while the device takes all at once
  float load() const {
    const uint64_t wgs = (uint64_t)nchunk * njw * ksegs;
    return wgs <= 512 ? (float)((wgs + 255) / 256) : (float)wgs / 256.0f;
  }
};

bool clamped_form(const SweepLaunch &L) {
  return L.cond_mode == BK_COND_REFERENCE || L.theta >= 0.0;
}

// What a pass takes, in us.  A single sweep and a pass by blocks are linear in
// the bricks (in thousands).  By strips a wave takes `alone` per plane where it
// has its SIMD to itself, the device `each` per plane and workgroup of a CU,
// and the memory `brick` per thousand bricks.  Fitted over 28 boxes of 8 to
// 262144 bricks, one to 80 an axis (errors up to 12 %, single sweeps of a few
// thousand bricks 25 %).  The form that the model takes is the fastest one or
// within 5 % of it in all but a few of the 28 boxes and 12 kinds.  Some of both
// sides, us a sweep (single / blocks / strips): 7-point FP64 8^3 bricks 4.7 /
// 2.7 / 6.6, 20^3 15.6 / 12.9 / 10.5, 64^3 411 / 376 / 155, 1x140x140 39 / 32 /
// 62; BF16 64^3 116 / 227 / 97; 13-point FP64 8^3 5.5 / 4.6 / 13, 16^3 11.0 / 14
// / 14, 64^3 434 / 900 / 289, FP32 8^3 6.0 / 4.1 / 10, 64^3 228 / 370 / 166.
struct Line {
  float at0, per_k;
};
struct Strip {
  float at0, alone, each, brick;  // at0 < 0: not built
};
struct PassModel {
  Line single;
  Line block[2];   // passes of 3 and 4 sweeps; radius 2: of 2
  Strip strip[2];
};
constexpr Strip kNoStrip = {-1.0f, 0.0f, 0.0f, 0.0f};
constexpr Line kNoLine = {-1.0f, 0.0f};
const PassModel kModel[4][3] = {
    // 7-point: FP64, FP32, BF16
    {{{4.07f, 1.56f}, {{6.32f, 4.6f}, {6.8f, 5.77f}},
      {{5.64f, 1.2f, 0.89f, 2.03f}, {5.6f, 1.52f, 1.17f, 2.31f}}},
     {{3.81f, 0.81f}, {{6.37f, 2.25f}, {6.68f, 3.06f}},
      {{5.93f, 1.0f, 0.71f, 1.11f}, {7.03f, 1.21f, 0.89f, 1.31f}}},
     {{4.08f, 0.48f}, {{6.45f, 2.61f}, {6.73f, 3.46f}},
      {{5.85f, 1.2f, 0.81f, 1.05f}, {8.01f, 1.41f, 1.04f, 1.41f}}}},
    // cond, values: FP64, FP32, BF16
    {{{4.96f, 1.53f}, {{6.7f, 5.73f}, {7.44f, 7.45f}},
      {{5.02f, 2.46f, 1.77f, 2.46f}, kNoStrip}},
     {{4.4f, 0.8f}, {{6.7f, 3.23f}, {7.07f, 4.91f}},
      {{6.08f, 2.05f, 1.3f, 1.83f}, {5.07f, 2.83f, 1.84f, 2.48f}}},
     {{4.57f, 0.54f}, {{6.8f, 3.81f}, {7.54f, 5.39f}},
      {kNoStrip, kNoStrip}}},
    // cond, clamped values: FP64, FP32, BF16
    {{{4.95f, 1.54f}, {{6.71f, 5.74f}, {7.42f, 7.45f}},
      {{4.02f, 2.14f, 1.54f, 2.19f}, {20.0f, 1.68f, 1.84f, 2.75f}}},
     {{4.38f, 0.81f}, {{6.68f, 3.21f}, {7.06f, 4.89f}},
      {{6.06f, 1.74f, 1.17f, 1.62f}, {10.79f, 2.13f, 1.53f, 2.04f}}},
     {{4.54f, 0.54f}, {{6.74f, 3.8f}, {7.51f, 5.39f}},
      {kNoStrip, kNoStrip}}},
    // 13-point: FP64, FP32, BF16
    {{{4.73f, 1.64f}, {{6.24f, 5.98f}, kNoLine},
      {{5.79f, 1.42f, 1.02f, 2.19f}, kNoStrip}},
     {{4.28f, 0.84f}, {{6.53f, 2.56f}, kNoLine},
      {{5.44f, 1.23f, 0.82f, 1.22f}, kNoStrip}},
     {{4.36f, 0.5f}, {{6.18f, 3.29f}, kNoLine},
      {kNoStrip, kNoStrip}}},
};

constexpr float kNever = 1e9f;

// The time of a pass of ts sweeps and whether it goes by blocks.
float pass_time(const SweepLaunch &L, const PlanView &P, int ts, bool &block) {
  const int form = L.stencil == BK_STAR13 ? kStar13 : L.stencil == BK_STAR7 ? kStar
                   : clamped_form(L) ? kCondPos : kCondRaw;
  const int dt = L.dtype == BK_F64 ? 0 : L.dtype == BK_F32 ? 1 : 2;
  const PassModel &m = kModel[form][dt];
  const float k = (float)P.ncovered * 1e-3f;
  block = false;
  if (ts == 1) return m.single.at0 + m.single.per_k * k;
  if ((ts == 2) != (form == kStar13)) return kNever;  // not built
  const int q = ts == 4;
  const float b = m.block[q].at0 + m.block[q].per_k * k;
  float s = kNever;
  if (m.strip[q].at0 >= 0.0f) {
    const Strips st(P, ts);
    const float planes = (float)P.box_nb[2] * 8.0f / (float)st.ksegs +
                         2.0f * (float)(ts * radius_of(form));
    s = m.strip[q].at0 + std::max(planes * std::max(m.strip[q].alone, m.strip[q].each * st.load()),
                                  m.strip[q].brick * k);
  }
  block = b <= s;
  return std::min(b, s);
}

}  // namespace

bool steps_by_blocks(const SweepLaunch &L, const PlanView &P, int ts) {
  bool block;
  (void)pass_time(L, P, ts, block);
  return block;
}

namespace {

// Strips of four FP64 sweeps with unclamped cond planes spill (0.75 ms a
// sweep against 0.22 with three), and single sweeps are the faster ones of
// BF16's cond and 13-point at every size (cond 0.62 us per thousand bricks and
// sweep by three against 0.54): not built.
template <class T, int TS, int FORM>
constexpr bool strip_built() {
  if (std::is_same<T, bf16>::value) return FORM == kStar;
  return !(std::is_same<T, double>::value && TS == 4 && FORM == kCondRaw);
}

template <class T, int TS, int FORM>
hipError_t launch_steps_t(const SweepLaunch &L, const PlanView &P, hipStream_t s) {
  using A = typename acc_of<T>::type;
  StepArgs<T> a;
  a.ids = P.box_ids;
  a.affine = P.box_affine;
  a.base = P.box_base;
  for (int q = 0; q < 3; ++q) a.stride[q] = P.box_stride[q];
  a.in = static_cast<const T *>(L.in);
  a.out = static_cast<T *>(L.out);
  a.in_step = L.in_step;
  a.out_step = L.out_step;
  a.nb0 = P.box_nb[0];
  a.nb1 = P.box_nb[1];
  a.nb2 = P.box_nb[2];
  a.cond_mode = L.cond_mode;
  a.theta = (A)L.theta;
  for (int q = 0; q < 13; ++q) a.c[q] = (A)L.coeff[q];
  a.nchunk = a.njg = a.njw = a.ksegs = 0;
  if (steps_by_blocks(L, P, TS)) {
    // half bricks while whole ones would leave half of the 256 CUs without a
    // workgroup (64 bricks: 1.43 us a sweep against 1.58; 216: 1.72 / 1.70)
    if (P.ncovered <= 128)
      hipLaunchKernelGGL((star_steps_block<T, TS, 4, FORM>), dim3(P.ncovered * 2), dim3(256), 0,
                         s, a);
    else
      hipLaunchKernelGGL((star_steps_block<T, TS, 8, FORM>), dim3(P.ncovered), dim3(256), 0, s,
                         a);
    return hipGetLastError();
  }
  if constexpr (strip_built<T, TS, FORM>()) {
    const Strips st(P, TS);
    a.nchunk = st.nchunk;
    a.njg = st.njg;
    a.njw = st.njw;
    a.ksegs = st.ksegs;
    const uint64_t nblk = (uint64_t)st.nchunk * st.njw * st.ksegs;
    if (nblk > 0x7fffffffull) return hipErrorInvalidValue;
    hipLaunchKernelGGL((strip_kernel<T, TS, FORM>()), dim3((uint32_t)nblk), dim3(256), 0, s, a);
    return hipGetLastError();
  }
  return hipErrorInvalidValue;
}

template <class T, int FORM>
hipError_t launch_steps_dt(const SweepLaunch &L, const PlanView &P, int ts, hipStream_t s) {
  switch (ts) {
    case 3: return launch_steps_t<T, 3, FORM>(L, P, s);
    case 4: return launch_steps_t<T, 4, FORM>(L, P, s);
    default: return hipErrorInvalidValue;
  }
}

template <class T>
hipError_t launch_steps_st(const SweepLaunch &L, const PlanView &P, int ts, hipStream_t s) {
  if (L.stencil == BK_STAR7) return launch_steps_dt<T, kStar>(L, P, ts, s);
  if (L.stencil == BK_STAR13)
    return ts == 2 ? launch_steps_t<T, 2, kStar13>(L, P, s) : hipErrorInvalidValue;
  if (L.stencil == BK_COND7)
    return clamped_form(L) ? launch_steps_dt<T, kCondPos>(L, P, ts, s)
                           : launch_steps_dt<T, kCondRaw>(L, P, ts, s);
  return hipErrorInvalidValue;
}

}  // namespace

bool steps_fit(const SweepLaunch &L, const PlanView &P) {
  if (!P.box_ids || (L.stencil != BK_STAR7 && L.stencil != BK_COND7 && L.stencil != BK_STAR13))
    return false;
  // both fields take 16-byte stores (single ones in BF16)
  const size_t es = L.dtype == BK_F64 ? 8 : L.dtype == BK_F32 ? 4 : 2;
  const uintptr_t bits = reinterpret_cast<uintptr_t>(L.in) | reinterpret_cast<uintptr_t>(L.out) |
                         (uintptr_t)(L.in_step * es) | (uintptr_t)(L.out_step * es);
  return es == 2 || bits % 16 == 0;
}

// Several sweeps per pass have to be 6 % faster than the model of single ones.
void steps_costs(const SweepLaunch &L, const PlanView &P, float cost[5]) {
  bool block;
  cost[0] = 0.0f;
  for (int ts = 1; ts <= 4; ++ts) cost[ts] = pass_time(L, P, ts, block);
  cost[1] *= 0.94f;
}

hipError_t launch_star_steps(const SweepLaunch &L, const PlanView &P, int ts, hipStream_t s) {
  switch (L.dtype) {
    case BK_F64: return launch_steps_st<double>(L, P, ts, s);
    case BK_F32: return launch_steps_st<float>(L, P, ts, s);
    case BK_BF16: return launch_steps_st<bf16>(L, P, ts, s);
    default: return hipErrorInvalidValue;
  }
}

}  // namespace bk
