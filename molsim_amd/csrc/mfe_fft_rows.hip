// mfe_fft_rows.hip -- the x passes of the 3D FFT (mfe_fft.hip): the r2c
// transform of the spread rows, read from the spreading tiles, and the c2r
// transform back, in registers (rows_fwd, rows_inv) where s1/2 has no prime
// factor above 7, else through LDS (fftx_fwd_rows, fftx_inv_rows).
#include <hip/hip_runtime.h>

#include <algorithm>

#include "mfe_fft_device.h"
#include "mfe_internal.h"

namespace mfe {
namespace {

// The spread mesh at point (x, y, z): the point's value in its own brick's
// spreading tile plus the low-side halo values of the next brick along each
// axis (at most 8 tiles), added in a fixed order.  Tiles are the bricks
// extended by order-1 points below (see k_spread).
template <typename R>
__device__ __forceinline__ R spread_point(const SysDev &V, const R *__restrict__ tiles, int x,
                                          int y, int z) {
  const SpmeGeom &g = V.sg;
  const int h = g.order - 1;
  const int E0 = g.B[0] + h, E1 = g.B[1] + h, E2 = g.B[2] + h;
  const int bc0 = fdiv(x, g.fB[0]), bc1 = fdiv(y, g.fB[1]), bc2 = fdiv(z, g.fB[2]);
  const int l0 = x - bc0 * g.B[0], l1 = y - bc1 * g.B[1], l2 = z - bc2 * g.B[2];
  R acc = R(0);
  for (int dz = 0; dz < 2; ++dz) {
    if (dz && l2 < g.B[2] - h) break;
    const int tz = dz ? (bc2 + 1 == g.nb[2] ? 0 : bc2 + 1) : bc2;
    const int ez = l2 + h - dz * g.B[2];
    for (int dy = 0; dy < 2; ++dy) {
      if (dy && l1 < g.B[1] - h) break;
      const int ty = dy ? (bc1 + 1 == g.nb[1] ? 0 : bc1 + 1) : bc1;
      const int ey = l1 + h - dy * g.B[1];
      for (int dx = 0; dx < 2; ++dx) {
        if (dx && l0 < g.B[0] - h) break;
        const int tx = dx ? (bc0 + 1 == g.nb[0] ? 0 : bc0 + 1) : bc0;
        const int ex = l0 + h - dx * g.B[0];
        const int t = tx + g.nb[0] * (ty + g.nb[1] * tz);
        acc += tiles[(size_t)t * (E0 * E1 * E2) + (ez * E1 + ey) * E0 + ex];
      }
    }
  }
  return acc;
}

// The rows are read from the spreading tiles (the spread mesh is never
// stored).
template <typename R>
__global__ void __launch_bounds__(256) k_fft_x_fwd(const SysDev *__restrict__ sys) {
  const SysDev &V = sys[blockIdx.z];
  // neighbouring rows (which read the same spreading tiles) on one XCD
  const int blk = xcd_block(blockIdx.x, gridDim.x);
  if (V.cx.ns || blk >= V.fx_nblk) return;
  extern __shared__ char smem[];
  const R *__restrict__ tiles = (const R *)V.spread_tiles;
  const int nrows = V.sg.s[1] * V.sg.s[2], row0 = blk * V.fx_rpb;
  fftx_fwd_rows<R>(V, row0, min(V.fx_rpb, nrows - row0), V.fx_rpb, smem,
                   [&](int x, int y, int z) { return spread_point<R>(V, tiles, x, y, z); });
}

template <typename R>
__global__ void __launch_bounds__(256) k_fft_x_inv(const SysDev *__restrict__ sys) {
  const SysDev &V = sys[blockIdx.z];
  // neighbouring rows (which the y inverse wrote together) on one XCD
  const int blk = xcd_block(blockIdx.x, gridDim.x);
  if (V.cx.ns || blk >= V.fx_nblk) return;
  extern __shared__ char smem[];
  const int nrows = V.sg.s[1] * V.sg.s[2], row0 = blk * V.fx_rpb;
  fftx_inv_rows<R>(V, row0, min(V.fx_rpb, nrows - row0), V.fx_rpb, smem);
}

// The spread rows of the x forward pass (spread_point's sums in its order)
// read with every load in flight: a row's tile rows -- its own brick's, and
// the next brick's along y and z where the row lies in their low-side halo
// -- are found once per row, a point's two places in them (own brick and
// the next along x) once per point, and the up to eight loads of four
// points are issued together.  spread_point's branches made every load wait
// for the one before: the x forward pass at 128^3 FP32 21.5 -> 17.2 us (of
// which the reading of 21^3-point tiles for 16^3 points is about half),
// 240^3 149 -> 84, FP64 128^3 32 -> 18.9.
constexpr int kRowThreads = 256;
template <typename R>
__device__ __forceinline__ void load_spread_rows(const SysDev &V, int row0, int nr, int ld,
                                                 int4 *info, R *ar) {
  const SpmeGeom &g = V.sg;
  const R *__restrict__ tiles = (const R *)V.spread_tiles;
  const int h = g.order - 1, s1 = g.s[0], s2 = g.s[1];
  const int E0 = g.B[0] + h, E1 = g.B[1] + h, E2 = g.B[2] + h, E3 = E0 * E1 * E2;
  for (int r = threadIdx.x; r < nr; r += blockDim.x) {
    const int row = row0 + r, z = fdiv(row, V.f_s2), y = row - z * s2;
    const int by = fdiv(y, g.fB[1]), bz = fdiv(z, g.fB[2]);
    const int ly = y - by * g.B[1], lz = z - bz * g.B[2];
    const int by1 = by + 1 == g.nb[1] ? 0 : by + 1, bz1 = bz + 1 == g.nb[2] ? 0 : bz + 1;
    const bool hy = ly >= g.B[1] - h, hz = lz >= g.B[2] - h;
    // places of x = 0 in the tile rows (dz, dy) = 00, 01, 10, 11
    auto at = [&](int ty, int tz, int ey, int ez) {
      return (tz * g.nb[1] + ty) * g.nb[0] * E3 + (ez * E1 + ey) * E0 + h;
    };
    const int ey = ly + h, ez = lz + h;
    int4 o;
    o.x = at(by, bz, ey, ez);
    o.y = hy ? at(by1, bz, ey - g.B[1], ez) : -1;
    o.z = hz ? at(by, bz1, ey, ez - g.B[2]) : -1;
    o.w = hy && hz ? at(by1, bz1, ey - g.B[1], ez - g.B[2]) : -1;
    info[r] = o;
  }
  __syncthreads();
  constexpr int kU = 4;
  const int total = nr * s1;
  for (int e0 = threadIdx.x; e0 < total; e0 += kU * blockDim.x) {
    R v[kU][8];
    int dst[kU];
#pragma unroll
    for (int u = 0; u < kU; ++u) {
      const int e = e0 + u * blockDim.x;
      const bool on = e < total;
      const int r = on ? fdiv(e, V.f_s1) : 0, x = on ? e - r * s1 : 0;
      const int bx = fdiv(x, g.fB[0]), lx = x - bx * g.B[0];
      const bool hx = lx >= g.B[0] - h;
      const int xm = bx * E3 + lx, xh = (bx + 1 == g.nb[0] ? 0 : bx + 1) * E3 + lx - g.B[0];
      const int4 o = info[r];
      const int off[4] = {o.x, o.y, o.z, o.w};
      dst[u] = on ? 2 * (r * ld) + x : -1;
#pragma unroll
      for (int s = 0; s < 4; ++s) {
        v[u][2 * s] = R(0);
        v[u][2 * s + 1] = R(0);
        if (on && off[s] >= 0) {
          v[u][2 * s] = tiles[(size_t)(unsigned)(off[s] + xm)];
          if (hx) v[u][2 * s + 1] = tiles[(size_t)(unsigned)(off[s] + xh)];
        }
      }
    }
#pragma unroll
    for (int u = 0; u < kU; ++u) {
      R acc = R(0);
#pragma unroll
      for (int k = 0; k < 8; ++k) acc += v[u][k];
      if (dst[u] >= 0) ar[dst[u]] = acc;
    }
  }
  __syncthreads();
}

// The x passes in registers (rows_fwd, rows_inv).  Inverse: 128^3 FP32 9.9 ->
// 7.5 us (17 MB, 2.2 TB/s; bound by the latency of its one round trip),
// 240^3 58 -> 28; FP64 128^3 14 -> 10.
template <typename R>
__global__ void __launch_bounds__(kRowThreads) k_row_fwd(const SysDev *__restrict__ sys) {
  const SysDev &V = sys[blockIdx.z];
  const RowPlan &p = V.cx;
  // neighbouring rows (which read the same spreading tiles) on one XCD
  const int blk = xcd_block(blockIdx.x, gridDim.x);
  if (!p.ns || blk >= p.nblk) return;
  extern __shared__ __align__(16) char smem[];
  const int nrows = V.sg.s[1] * V.sg.s[2], row0 = blk * p.nr, nr = min(p.nr, nrows - row0);
  Twiddle<R> *twh = reinterpret_cast<Twiddle<R> *>(smem), *twf = twh + p.m;
  int4 *info = reinterpret_cast<int4 *>(twf + 2 * p.m);
  cplx<R> *A = reinterpret_cast<cplx<R> *>(info + p.nr), *B = A + p.nr * p.ld;
  stage_twiddles(twh, (const Twiddle<R> *)V.tw_half, p.m);
  stage_twiddles(twf, (const Twiddle<R> *)V.tw[0], 2 * p.m);
  load_spread_rows<R>(V, row0, nr, p.ld, info, reinterpret_cast<R *>(A));
  rows_fwd<R>(p, nr, A, B, twh, twf, (cplx<R> *)V.mesh_c + (size_t)row0 * V.hx);
}

template <typename R>
__global__ void __launch_bounds__(kRowThreads) k_row_inv(const SysDev *__restrict__ sys) {
  const SysDev &V = sys[blockIdx.z];
  const RowPlan &p = V.cx;
  // neighbouring rows (which the y inverse wrote together) on one XCD
  const int blk = xcd_block(blockIdx.x, gridDim.x);
  if (!p.ns || blk >= p.nblk) return;
  extern __shared__ __align__(16) char smem[];
  const int nrows = V.sg.s[1] * V.sg.s[2], row0 = blk * p.nr, nr = min(p.nr, nrows - row0);
  Twiddle<R> *twh = reinterpret_cast<Twiddle<R> *>(smem), *twf = twh + p.m;
  cplx<R> *A = reinterpret_cast<cplx<R> *>(twf + 2 * p.m), *B = A + p.nr * p.ld;
  stage_twiddles(twh, (const Twiddle<R> *)V.tw_half, p.m);
  stage_twiddles(twf, (const Twiddle<R> *)V.tw[0], 2 * p.m);
  __syncthreads();
  const int m = p.m;
  // a row of reals is a row of m (even, odd) pairs
  cplx<R> *real = (cplx<R> *)V.mesh_r + (size_t)row0 * m;
  rows_inv<R>(p, nr, A, B, twh, twf, (const cplx<R> *)V.mesh_c + (size_t)row0 * V.hx,
              [=](int k, int c, cplx<R> v) { real[(unsigned)(c * m + k)] = v; });
}

template <typename R>
int rows_per_block(int s1) {
  // two LDS buffers of rows*(s1/2+1) complex values, about 32 KB in all and
  // at most 16 rows; at FP64 about 48 KB and at most 32 rows (23 rows of 128
  // points measured faster there than 15, while FP32 is fastest at 16)
  constexpr bool f64 = sizeof(R) == 8;
  const int per_row = 2 * (s1 / 2 + 1) * (int)sizeof(cplx<R>);
  const int rows = ((f64 ? 48 : 32) * 1024) / per_row, cap = f64 ? 32 : 16;
  return rows < 1 ? 1 : (rows > cap ? cap : rows);
}

}  // namespace

// geometry of the rows through LDS
void fft_row_geometry(int prec, const int s[3], int *fx_rpb, int *fx_nblk, size_t *lds_fx) {
  const bool f = prec == MFE_PREC_MIXED;
  const size_t csz = f ? sizeof(cplx<float>) : sizeof(cplx<double>);
  const size_t tsz = f ? sizeof(Twiddle<float>) : sizeof(Twiddle<double>);
  int rpb = f ? rows_per_block<float>(s[0]) : rows_per_block<double>(s[0]);
  // the rows and the twiddles within 64 KB of LDS
  while (rpb > 1 && 2 * (size_t)rpb * (s[0] / 2 + 1) * csz + (size_t)(s[0] / 2 + s[0]) * tsz >
                        64 * 1024)
    --rpb;
  *fx_rpb = rpb;
  *fx_nblk = (s[1] * s[2] + rpb - 1) / rpb;
  // two row buffers, then the half- and full-length twiddles
  *lds_fx = 2 * (size_t)rpb * (s[0] / 2 + 1) * csz + (size_t)(s[0] / 2 + s[0]) * tsz;
}

// Rows per block: 16 (8 on long rows, within the column passes' LDS), and
// threads for one butterfly each of the first radix.
RowPlan row_plan(int prec, const int s[3], const int B[3], int order) {
  const bool f = prec == MFE_PREC_MIXED;
  const size_t csz = f ? sizeof(cplx<float>) : sizeof(cplx<double>);
  const size_t tsz = f ? sizeof(Twiddle<float>) : sizeof(Twiddle<double>);
  RowPlan p{};
  const int m = s[0] / 2;
  if (!fft_radices(m, 8, &p.ns, p.r)) return p;
  // tile places of the forward pass as 32-bit offsets
  double tiles = 1.0;
  for (int a = 0; a < 3; ++a) tiles *= (double)s[a] * (B[a] + order - 1) / B[a];
  if (tiles >= 2147483648.0) {
    p.ns = 0;
    return p;
  }
  p.m = m;
  p.ld = m | 1;
  const size_t tab = 3 * (size_t)m * tsz, row = 2 * (size_t)p.ld * csz + sizeof(int4);
  p.nr = 16;
  while (p.nr > 1 && tab + p.nr * row > kColLds) p.nr /= 2;
  if (tab + p.nr * row > kColLds) {
    p.ns = 0;
    return p;
  }
  p.nblk = (s[1] * s[2] + p.nr - 1) / p.nr;
  const int items = p.nr * (m / p.r[p.ns - 1]);
  p.nthr = std::min(kRowThreads, std::max(64, (items + 63) / 64 * 64));
  p.lds = (int)(tab + p.nr * row);
  for (int k = 0; k < p.ns; ++k) p.f_nb[k] = make_fastdiv(m / p.r[k]);
  p.f_pair = make_fastdiv(m / p.r[p.ns - 1] / 2 + 1);
  return p;
}

// The forward pass on the mixed path takes kRowThreads threads whatever the
// butterflies need, for its tile loads (four points of a thread in flight),
// where the launch has few blocks: 128^3 16.4 -> 13.1 us, 64^3 8.9 -> 7.0,
// 70^3 9.8 -> 8.2, 240^3 no change (512 threads: 17.0, 6.6, 7.7 and 94.9
// against 82.7).  Launches that fill the chip several times over lose by it
// (a batch of 96 replicas of 36^3 4% of its step); FP64 128^3 19.8 either way.
constexpr long long kFewRowBlocks = 2048;
void fft_x_forward(const Group &g) {
#define MFE_X(T, ROW, LDS_ROWS, THR)                                                          \
  do {                                                                                        \
    if (g.cx_blocks)                                                                          \
      hipLaunchKernelGGL(ROW<T>, dim3(g.cx_blocks, 1, g.R), dim3(THR), g.lds_cx, g.stream,    \
                         g.d);                                                                \
    if (g.fx_blocks)                                                                          \
      hipLaunchKernelGGL(LDS_ROWS<T>, dim3(g.fx_blocks, 1, g.R), dim3(256), g.lds_fx,         \
                         g.stream, g.d);                                                      \
  } while (0)
  if (g.prec == MFE_PREC_MIXED) {
    const bool few = (long long)g.cx_blocks * g.R <= kFewRowBlocks;
    MFE_X(float, k_row_fwd, k_fft_x_fwd, few ? kRowThreads : g.cx_thr);
  } else {
    MFE_X(double, k_row_fwd, k_fft_x_fwd, g.cx_thr);
  }
}
void fft_x_inverse(const Group &g) {
  if (g.prec == MFE_PREC_MIXED) MFE_X(float, k_row_inv, k_fft_x_inv, g.cx_thr);
  else MFE_X(double, k_row_inv, k_fft_x_inv, g.cx_thr);
#undef MFE_X
}
}  // namespace mfe
