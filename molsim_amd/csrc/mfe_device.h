// mfe_device.h -- device helpers shared by the kernel translation units of
// libmfe (gfx950 only): minimum image, block reductions, lane exchanges,
// compensated sums, the spline pair term's weights, CardinalBSpline, mesh
// coordinates and the spreading accumulators.
#pragma once

#include <hip/hip_runtime.h>

#include "mfe_internal.h"

namespace mfe {
namespace {

constexpr int kBlock = 256;

// ---------------------------------------------------------------- helpers
// PBCr2 for the box (Src/molaux.F90:159-182): one shift per axis, then
// r2 = dx**2 + dy**2 + dz**2 summed left to right without fusion, so that
// list membership is decided on the reference's FP64 value.
__device__ __forceinline__ double pbcr2(double &dx, double &dy, double &dz,
                                        const Box &b) {
#pragma clang fp contract(off)
  if (fabs(dx) > b.L2[0]) dx = dx - copysign(b.L[0], dx);
  if (fabs(dy) > b.L2[1]) dy = dy - copysign(b.L[1], dy);
  if (fabs(dz) > b.L2[2]) dz = dz - copysign(b.L[2], dz);
  double r2 = dx * dx;
  r2 = r2 + dy * dy;
  r2 = r2 + dz * dz;
  return r2;
}

// The partner value of an FP64 register in a lane quad, by DPP (no LDS):
// kXor1 swaps lanes 0<->1 and 2<->3, kXor2 swaps 0<->2 and 1<->3 -- the
// exchanges of __shfl_xor(x, 1 or 2) within a quad.  Every lane of the
// wavefront must be active.
constexpr int kXor1 = 0xB1;  // quad_perm [1, 0, 3, 2]
constexpr int kXor2 = 0x4E;  // quad_perm [2, 3, 0, 1]
template <int CTRL>
__device__ __forceinline__ double quad_swap(double x) {
  const int lo = __builtin_amdgcn_mov_dpp(__double2loint(x), CTRL, 0xF, 0xF, false);
  const int hi = __builtin_amdgcn_mov_dpp(__double2hiint(x), CTRL, 0xF, 0xF, false);
  return __hiloint2double(hi, lo);
}

// Sum over the wavefront of an FP64 value, by DPP exchanges inside each row
// of 16 lanes (quads, half rows, rows) and lane reads across the four rows:
// no LDS round trips (a shuffle tree of FP64 takes twelve).  Every lane of
// the wavefront must be active; every lane gets the sum.
constexpr int kHalfMirror = 0x141;  // lane 7 - l of each 8
constexpr int kMirror = 0x140;      // lane 15 - l of each 16
__device__ __forceinline__ double read_lane(double x, int lane) {
  return __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(x), lane),
                          __builtin_amdgcn_readlane(__double2loint(x), lane));
}
__device__ __forceinline__ double wave_sum(double x) {
  x += quad_swap<kXor1>(x);
  x += quad_swap<kXor2>(x);
  x += quad_swap<kHalfMirror>(x);
  x += quad_swap<kMirror>(x);
  return (read_lane(x, 0) + read_lane(x, 16)) + (read_lane(x, 32) + read_lane(x, 48));
}

// Block-wide sum (max) in a fixed order: wave_sum (for the maximum a shuffle
// tree) inside each wavefront, then the wavefront results in wavefront order.
// Every thread gets the result; sh needs one slot per wavefront.
__device__ __forceinline__ double block_sum(double v, double *sh) {
  v = wave_sum(v);
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  __syncthreads();
  if (lane == 0) sh[wave] = v;
  __syncthreads();
  double r = sh[0];
  for (int k = 1; k < (int)(blockDim.x >> 6); ++k) r += sh[k];
  return r;
}

__device__ __forceinline__ double block_max(double v, double *sh) {
  for (int w = 32; w > 0; w >>= 1) v = fmax(v, __shfl_down(v, w, 64));
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  __syncthreads();
  if (lane == 0) sh[wave] = v;
  __syncthreads();
  double r = sh[0];
  for (int k = 1; k < (int)(blockDim.x >> 6); ++k) r = fmax(r, sh[k]);
  return r;
}

// out[c] (+)= sum over rows b of part[b * ncol + c], c < cols, in a fixed
// order: a block of 1024 threads takes 16 columns (128 bytes of a row) in 64
// slices of rows, eight loads in flight per thread, then the slices in order.
// 391 columns of 1032 rows: 6 us (a thread per column walked the rows one
// load after another: 63-101 us).  Grid: (cols + 15) / 16 blocks.
constexpr int kSumCols = 16, kSumThreads = 1024;
__device__ __forceinline__ void column_sums(const double *__restrict__ part, int rows, int ncol,
                                            int cols, double *__restrict__ out, bool add) {
  constexpr int kSlices = kSumThreads / kSumCols, kU = 8;
  __shared__ double sh[kSlices][kSumCols];
  const int cl = threadIdx.x % kSumCols, sl = threadIdx.x / kSumCols;
  const int c = blockIdx.x * kSumCols + cl;
  double s = 0.0;
  if (c < cols) {
    for (int b0 = sl; b0 < rows; b0 += kU * kSlices) {
      double v[kU];
#pragma unroll
      for (int u = 0; u < kU; ++u) {
        const int b = b0 + u * kSlices;
        v[u] = b < rows ? part[(size_t)b * ncol + c] : 0.0;
      }
#pragma unroll
      for (int u = 0; u < kU; ++u) s += v[u];
    }
  }
  sh[sl][cl] = s;
  __syncthreads();
  if (sl == 0 && c < cols) {
    double t = 0.0;
    for (int k = 0; k < kSlices; ++k) t += sh[k][cl];
    out[c] = add ? out[c] + t : t;
  }
}

// index of the pair of types i and j (Set_iptpt order: j >= i, j fastest)
__device__ __forceinline__ int pair_index(int i, int j, int npt) {
  const int a = min(i, j), b = max(i, j);
  return a * npt - a * (a - 1) / 2 + b - a;
}

struct KahanF {
  float s = 0.f, c = 0.f;
  __device__ __forceinline__ void add(float v) {
    float y = v - c;
    float t = s + y;
    c = (t - s) - y;
    s = t;
  }
  __device__ __forceinline__ double value() const { return (double)s - (double)c; }
};

// a / D for a small integer D, as the reference divides.  Powers of two
// multiply exactly.  Otherwise the product with the rounded reciprocal is
// refined by one FMA step (q + (a - q D) / D), which gives the correctly
// rounded quotient: multiplying by RN(1/3) or RN(1/5) alone rounds every
// quotient the same way, and on the FP32 path that bias (5e-8 per axis at
// order 6, so 1.4e-7 on the spread charge and 3e-7 on the reciprocal
// energy) does not average out over the mesh.
template <typename R, int D>
__device__ __forceinline__ R div_small(R a) {
  constexpr R inv = R(1.0 / D);
  if constexpr ((D & (D - 1)) == 0) {
    return a * inv;
  } else if constexpr (sizeof(R) == 4) {
    const float q = a * inv;
    const float r = __builtin_fmaf(-q, float(D), a);
    return __builtin_fmaf(r, inv, q);
  } else {
    const double q = a * inv;
    const double r = __builtin_fma(-q, double(D), a);
    return __builtin_fma(r, inv, q);
  }
}

// ------------------------------------------------- spline pair term
// Uniform cubic B-spline on knots r0 + k/dinv: on interval i (fraction f)
// the weights of coefficients i..i+3 are (1-f)^3/6, (3f^3-6f^2+4)/6,
// (-3f^3+3f^2+3f+1)/6, f^3/6 (de Boor, A Practical Guide to Splines, ch. IX),
// and their derivatives in f.
__device__ __forceinline__ bool knot_weights(double r, double r0, double dinv, int nknot,
                                             int &i, double w[4], double dw[4]) {
  const double x = (r - r0) * dinv;
  if (!(x >= 0.0) || !(x < (double)(nknot - 3))) return false;
  i = (int)x;
  const double f = x - i, f2 = f * f, f3 = f2 * f, g = 1.0 - f;
  w[0] = div_small<double, 6>(g * g * g);
  w[1] = div_small<double, 6>(3.0 * f3 - 6.0 * f2 + 4.0);
  w[2] = div_small<double, 6>(-3.0 * f3 + 3.0 * f2 + 3.0 * f + 1.0);
  w[3] = div_small<double, 6>(f3);
  dw[0] = -0.5 * g * g;
  dw[1] = 1.5 * f2 - 2.0 * f;
  dw[2] = -1.5 * f2 + f + 0.5;
  dw[3] = 0.5 * f2;
  return true;
}

// CardinalBSpline (Src/mollib.F90:1629-1683) at fraction x in [0,1), without
// its divisions: v[i] is (ORDER-1)! times the weight of grid point kmax - i,
// d[i] (ORDER-2)! times its derivative.  The recursion's stage n divides by
// n - 1; here the whole divisor is applied once, in FP64, to what the
// weights are summed to (kSplineScale), exactly enough that no rounded
// reciprocal biases the weights.  A value is a multiplication and an FMA:
// at order 6 three axes take about 150 operations, 380 with a correctly
// rounded quotient at each stage (200k ions: FP64 gather 41 -> 34.9 us with
// the same lanes, spreading 23.1 -> 21.4 us, bound by its LDS adds).
template <typename R, int ORDER, int N>
__device__ __forceinline__ void bspline_stage(const R *up, const R *dn, R *v, R *last) {
  if constexpr (N <= ORDER) {
#pragma unroll
    for (int i = 0; i < N - 1; ++i) last[i] = v[i];
    v[0] = up[0] * last[0];
#pragma unroll
    for (int i = 1; i <= N - 2; ++i) v[i] = up[i] * last[i] + dn[N - i] * last[i - 1];
    v[N - 1] = dn[1] * last[N - 2];
    bspline_stage<R, ORDER, N + 1>(up, dn, v, last);
  }
}

template <typename R, int ORDER>
__device__ __forceinline__ void bspline(R x, R *v, R *d) {
  // x + i and i - x, the factors of every stage
  R up[ORDER], dn[ORDER], last[ORDER];
#pragma unroll
  for (int i = 0; i < ORDER; ++i) {
    up[i] = R(i) + x;
    dn[i] = R(i) - x;
    last[i] = R(0);
    v[i] = R(0);
  }
  v[0] = x;
  v[1] = dn[1];
  bspline_stage<R, ORDER, 3>(up, dn, v, last);
  if (d) {
    d[0] = last[0];
#pragma unroll
    for (int i = 1; i <= ORDER - 2; ++i) d[i] = last[i] - last[i - 1];
    d[ORDER - 1] = -last[ORDER - 2];
  }
}

// what a product of three of bspline's values, ND (0 or 1) of them derivatives, is to
// be multiplied by
constexpr double factorial(int n) { return n < 2 ? 1.0 : n * factorial(n - 1); }
template <int ORDER, int ND>
constexpr double kSplineScale =
    1.0 / ((ND > 0 ? factorial(ORDER - 2) : factorial(ORDER - 1)) *
           factorial(ORDER - 1) * factorial(ORDER - 1));

__device__ __forceinline__ void mesh_coords(const double *r, const SpmeGeom &g,
                                            int mm[3], double fr[3]) {
  for (int m = 0; m < 3; ++m) {
    const double u = g.dkdr[m] * r[m];
    const double f = floor(u);
    fr[m] = u - f;
    int k = (int)f % g.s[m];
    mm[m] = k < 0 ? k + g.s[m] : k;
  }
}

// LDS accumulator of the spreading: exact 64-bit fixed point (2^-32) for
// the mixed path, so the sum does not depend on the order of the adds;
// FP64 LDS atomics for the FP64 path.  What is added is scale * v: on the
// mixed path the fixed-point value is scale * v * 2^32 + 1.5 * 2^52 in FP64
// (one FMA; it rounds once to an integer because |scale * v| * 2^32 < 2^51),
// whose low mantissa bits minus those of 1.5 * 2^52 are the two's-complement
// integer; on the FP64 path the scale goes into what the v are products of
// (pre).
template <typename R>
struct SpreadAcc;
template <>
struct SpreadAcc<float> {
  typedef unsigned long long T;
  static __device__ __forceinline__ float pre(float q, double) { return q; }
  static __device__ __forceinline__ void add(T *p, float v, double scale) {
    constexpr double kMagic = 6755399441055744.0;  // 1.5 * 2^52
    const double d = __fma_rn((double)v, 4294967296.0 * scale, kMagic);
    atomicAdd(p, (unsigned long long)__double_as_longlong(d) -
                     (unsigned long long)__double_as_longlong(kMagic));
  }
  static __device__ __forceinline__ float get(T v) {
    return (float)((double)(long long)v * (1.0 / 4294967296.0));
  }
};
template <>
struct SpreadAcc<double> {
  typedef double T;
  static __device__ __forceinline__ double pre(double q, double scale) { return q * scale; }
  static __device__ __forceinline__ void add(T *p, double v, double) { atomicAdd(p, v); }
  static __device__ __forceinline__ double get(T v) { return v; }
};

constexpr int kMaxOrder = 8;

// the spreading tile (z planes of SpmeGeom::plane values) written to global
// memory without the padding
template <typename R>
__device__ __forceinline__ void store_tile(const SpmeGeom &g, int E0, int E1, int E2,
                                           const typename SpreadAcc<R>::T *tile,
                                           R *__restrict__ out) {
  const int pad = g.plane - E0 * E1;
  for (int k = threadIdx.x; k < E0 * E1 * E2; k += blockDim.x) {
    const int z = pad ? fdiv(fdiv(k, g.fE[0]), g.fE[1]) : 0;
    out[k] = SpreadAcc<R>::get(tile[k + z * pad]);
  }
}

// one particle record in brick order: fraction (x, y, z) and charge
template <typename R>
struct Rec4 {
  R x, y, z, q;
};
__device__ __forceinline__ Rec4<float> load_rec(const float *__restrict__ p) {
  const float4 v = *reinterpret_cast<const float4 *>(p);
  return {v.x, v.y, v.z, v.w};
}
__device__ __forceinline__ Rec4<double> load_rec(const double *__restrict__ p) {
  const double2 a = reinterpret_cast<const double2 *>(p)[0];
  const double2 b = reinterpret_cast<const double2 *>(p)[1];
  return {a.x, a.y, b.x, b.y};
}

}  // namespace
}  // namespace mfe
