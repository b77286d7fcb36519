// mfe_fft.hip -- the 3D FFT of SPMFFTRec (Src/energy.F90:6525-6587) on the
// mesh of UEwaldRecSPM, in FFTW's unnormalised r2c/c2r convention:
// real mesh [s3][s2][s1] (Fortran Qmesh(s1,s2,s3)) <-> complex mesh
// [s3][s2][s1/2+1].
//
// Five passes, each reading and writing the mesh once:
//   x forward  : r2c of every x row through a complex FFT of half length
//   y forward  : complex FFT along y for tiles of kx columns
//   conv       : z forward, Green function (meshfac) with the FP64 energy
//                and virial sums of the reference's CalcGIF loop, z inverse
//                -- the z transform pair is fused around the pointwise
//                product, so the mesh is not written between them
//   y inverse, x inverse (c2r)
// The transforms run in registers with one LDS exchange per radix after the
// first (col_fft, rows_fwd, rows_inv) where the length has no prime factor
// above 7; other lengths are mixed-radix Stockham FFTs staged in LDS.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "mfe_fft_device.h"
#include "mfe_internal.h"

namespace mfe {
namespace {

// ------------------------------------------------------------ pass kernels
template <typename R>
__global__ void __launch_bounds__(256) k_fft_y(const SysDev *__restrict__ sys, int inv) {
  const SysDev &V = sys[blockIdx.z];
  if (V.cy.ns) return;
  // the tiles of one z plane share the cache lines of its rows: the blocks
  // of a contiguous range of planes go to one XCD
  const int L = xcd_block(blockIdx.y * gridDim.x + blockIdx.x, gridDim.x * gridDim.y);
  const int bx = L % gridDim.x, z = L / gridDim.x;
  if (bx >= V.fy_nbx || z >= V.sg.s[2]) return;
  extern __shared__ char smem[];
  ffty_tile<R>(V, bx, z, inv, smem);
}

// The y pass in registers.  Columns (z, kx) are numbered z hx + kx over the
// whole mesh and a block takes 1 << lgT consecutive ones (128 bytes of each
// row), so every block but the last is full whatever hx is, and loads go
// straight to the first radix: the mesh is in flight at once.  Bound by the
// latency of one load and one store round trip of that; XCD-contiguous
// blocks, as the rows of a plane share cache lines.  FP32 128^3 13.3 -> 8.1
// us (17 MB in and out, 4.2 TB/s), 240^3 74 -> 26; FP64 128^3 19.4 -> 12.3.
constexpr int kColThreads = 256;
template <typename R, bool INV>
__global__ void __launch_bounds__(kColThreads) k_col_y(const SysDev *__restrict__ sys) {
  const SysDev &V = sys[blockIdx.z];
  const ColPlan &p = V.cy;
  const int blk = xcd_block(blockIdx.x, gridDim.x);
  if (!p.ns || blk >= p.nblk) return;
  extern __shared__ __align__(16) char smem[];
  const int n = p.n, hx = V.hx, col0 = blk << p.lgT, nt = min(1 << p.lgT, p.ncol - col0);
  Twiddle<R> *tw = reinterpret_cast<Twiddle<R> *>(smem);
  cplx<R> *A = reinterpret_cast<cplx<R> *>(tw + n), *B = A + ((size_t)n << p.lgT);
  stage_twiddles(tw, (const Twiddle<R> *)V.tw[1], n);
  // a thread keeps its column over all items (blockDim a multiple of T)
  const int col = col0 + min((int)threadIdx.x & ((1 << p.lgT) - 1), nt - 1);
  const int z = fdiv(col, V.f_hx);
  cplx<R> *base = (cplx<R> *)V.mesh_c + (size_t)z * n * hx + (col - z * hx);
  col_fft<R, INV>(
      p, nt, A, B, tw, [=](int y, int) { return base[(unsigned)(y * hx)]; },
      [=](int y, int, cplx<R> v) { base[(unsigned)(y * hx)] = v; });
}

// The thread's energy and virial terms of a convolution block into its
// partials: shuffle trees in each wavefront, then the wavefronts in order.
__device__ __forceinline__ void conv_partials(const SysDev &V, int blk, double esum,
                                              double vsum) {
  __shared__ double red[2][kColThreads / 64];
  for (int w = 32; w > 0; w >>= 1) {
    esum += __shfl_down(esum, w, 64);
    vsum += __shfl_down(vsum, w, 64);
  }
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  if (lane == 0) {
    red[0][wave] = esum;
    red[1][wave] = vsum;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    double e = red[0][0], v = red[1][0];
    for (int k = 1; k < (int)(blockDim.x >> 6); ++k) {
      e += red[0][k];
      v += red[1][k];
    }
    double *__restrict__ part = V.part + V.off_conv;
    part[blk] = e;
    part[V.nblk_conv + blk] = v;
  }
}

template <typename R>
__global__ void __launch_bounds__(256) k_fft_conv(const SysDev *__restrict__ sys, int energy) {
  const SysDev &V = sys[blockIdx.z];
  if (V.cz.ns) return;
  // the tiles of one y line share the cache lines of its rows: the blocks
  // of a contiguous range of lines go to one XCD
  const int L = xcd_block(blockIdx.y * gridDim.x + blockIdx.x, gridDim.x * gridDim.y);
  const int bx = L % gridDim.x, y = L / gridDim.x;
  if (bx >= V.fz_nbx || y >= V.sg.s[1]) return;
  extern __shared__ char smem[];
  double esum = 0.0, vsum = 0.0;
  fftconv_tile<R>(V, bx, y, energy, smem, esum, vsum);
  if (energy) conv_partials(V, y * V.fz_nbx + bx, esum, vsum);
}

// The z pass in registers: forward, Green function (fftconv_tile's terms),
// inverse, over columns (y, kx), which are contiguous in each z plane; the
// product is applied between the forward transform's last radix and the
// inverse's first, in the same registers, so the pair takes two LDS
// exchanges of 16 x 8 points in place of sixteen LDS passes.  FP32 128^3
// 23.4 -> 15.8 us, 240^3 129 -> 49; FP64 128^3 37.4 -> 26.5 (its FP64 Green
// function and two transforms per load).
template <typename R>
__global__ void __launch_bounds__(kColThreads) k_col_conv(const SysDev *__restrict__ sys,
                                                          int energy) {
  const SysDev &V = sys[blockIdx.z];
  const ColPlan &p = V.cz;
  const int blk = xcd_block(blockIdx.x, gridDim.x);
  if (!p.ns || blk >= p.nblk) return;
  extern __shared__ __align__(16) char smem[];
  const int s1 = V.sg.s[0], s2 = V.sg.s[1], n = p.n, hx = V.hx, n2 = n / 2 + 1;
  const int col0 = blk << p.lgT, nt = min(1 << p.lgT, p.ncol - col0);
  const SpmeAxes &ax = V.ax;
  Twiddle<R> *tw = reinterpret_cast<Twiddle<R> *>(smem);
  double *gz = reinterpret_cast<double *>(tw + n), *kkz = gz + n2;
  cplx<R> *A = reinterpret_cast<cplx<R> *>(kkz + n2), *B = A + ((size_t)n << p.lgT);
  stage_twiddles(tw, (const Twiddle<R> *)V.tw[2], n);
  for (int k = threadIdx.x; k < n2; k += blockDim.x) {
    gz[k] = ax.g[2][k];
    kkz[k] = ax.kk[2][k];
  }
  // a single-stage plan reads the tables before any exchange's barrier
  if (p.ns == 1) __syncthreads();
  const int col = col0 + min((int)threadIdx.x & ((1 << p.lgT) - 1), nt - 1);
  const int y = fdiv(col, V.f_hx), nx = col - y * hx, ny = min(y, s2 - y);
  const double gxy = ax.fac0 * ax.g[0][nx] * ax.g[1][ny], kkxy = ax.kk[0][nx] + ax.kk[1][ny];
  const double w = (nx == 0 || 2 * nx == s1) ? 0.5 : 1.0;
  const unsigned zstride = (unsigned)(s2 * hx);
  cplx<R> *base = (cplx<R> *)V.mesh_c + col;
  double esum = 0.0, vsum = 0.0;
  col_conv<R>(
      p, nt, A, B, tw, [=](int z, int) { return base[(size_t)z * zstride]; },
      [&](int z, int, cplx<R> v) -> cplx<R> {
        const int nz = min(z, n - z);
        const double m2 = kkxy + kkz[nz];
        const double mf = m2 > 0.0 ? gxy * gz[nz] / m2 : 0.0;
        if (energy) {
          const double q2 = (double)v.x * (double)v.x + (double)v.y * (double)v.y;
          esum += w * q2 * mf;
          vsum -= w * q2 * (1.0 + 2.0 * m2 * ax.expf) * mf;
        }
        const R mfr = (R)mf;
        return {v.x * mfr, v.y * mfr};
      },
      [=](int z, int, cplx<R> v) { base[(size_t)z * zstride] = v; });
  if (energy) conv_partials(V, blk, esum, vsum);
}

// the z forward transform into out (the MC trial moves' kept spectrum,
// FP64 on both precision paths, so that accepted changes add to it without
// FP32 rounding)
template <typename R>
__global__ void __launch_bounds__(256) k_fft_z_fwd(const SysDev *__restrict__ sys, void *out) {
  const SysDev &V = sys[blockIdx.z];
  if (V.cz.ns) return;
  const int L = xcd_block(blockIdx.y * gridDim.x + blockIdx.x, gridDim.x * gridDim.y);
  const int bx = L % gridDim.x, y = L / gridDim.x;
  if (bx >= V.fz_nbx || y >= V.sg.s[1]) return;
  extern __shared__ char smem[];
  fftz_fwd_tile<R, double>(V, bx, y, (cplx<double> *)out, smem);
}
template <typename R>
__global__ void __launch_bounds__(kColThreads) k_col_z_fwd(const SysDev *__restrict__ sys,
                                                           void *out) {
  const SysDev &V = sys[blockIdx.z];
  const ColPlan &p = V.cz;
  const int blk = xcd_block(blockIdx.x, gridDim.x);
  if (!p.ns || blk >= p.nblk) return;
  extern __shared__ __align__(16) char smem[];
  const int n = p.n, col0 = blk << p.lgT, nt = min(1 << p.lgT, p.ncol - col0);
  Twiddle<R> *tw = reinterpret_cast<Twiddle<R> *>(smem);
  cplx<R> *A = reinterpret_cast<cplx<R> *>(tw + n), *B = A + ((size_t)n << p.lgT);
  stage_twiddles(tw, (const Twiddle<R> *)V.tw[2], n);
  const int col = col0 + min((int)threadIdx.x & ((1 << p.lgT) - 1), nt - 1);
  const cplx<R> *base = (const cplx<R> *)V.mesh_c + col;
  cplx<double> *obase = (cplx<double> *)out + col;
  const unsigned zstride = (unsigned)p.ncol;
  col_fft<R, false>(
      p, nt, A, B, tw, [=](int z, int) { return base[(size_t)z * zstride]; },
      [=](int z, int, cplx<R> v) {
        obase[(size_t)z * zstride] = cplx<double>{(double)v.x, (double)v.y};
      });
}

inline int tile_width(int hx, int target) {
  const int ntiles = (hx + target - 1) / target;
  return (hx + ntiles - 1) / ntiles;
}

template <typename R>
int tile_target(int n) {
  const int per_col = 2 * (n + 1) * (int)sizeof(cplx<R>);
  int t = (32 * 1024) / per_col;
  return t < 1 ? 1 : (t > 16 ? 16 : t);
}

}  // namespace

void fft_geometry(int prec, const int s[3], int *fx_rpb, int *fx_nblk, int *fy_T, int *fy_nbx,
                  int *fz_T, int *fz_nbx, size_t *lds_fx, size_t *lds_fy, size_t *lds_fz) {
  const bool f = prec == MFE_PREC_MIXED;
  const size_t csz = f ? sizeof(cplx<float>) : sizeof(cplx<double>);
  const size_t tsz = f ? sizeof(Twiddle<float>) : sizeof(Twiddle<double>);
  const int hx = s[0] / 2 + 1;
  fft_row_geometry(prec, s, fx_rpb, fx_nblk, lds_fx);
  const int Ty = tile_width(hx, f ? tile_target<float>(s[1]) : tile_target<double>(s[1]));
  *fy_T = Ty;
  *fy_nbx = (hx + Ty - 1) / Ty;
  *lds_fy = 2 * (size_t)Ty * (s[1] + 1) * csz + (size_t)s[1] * tsz;
  const int Tz = tile_width(hx, f ? tile_target<float>(s[2]) : tile_target<double>(s[2]));
  *fz_T = Tz;
  *fz_nbx = (hx + Tz - 1) / Tz;
  *lds_fz = 2 * (size_t)Tz * (s[2] + 1) * csz + (size_t)s[2] * tsz;
}

// n as at most three radices in descending order, the last (smallest) at
// most `last`: the fewest, then the smallest largest one; false when n has
// none
bool fft_radices(int n, int last, int *ns, int r[3]) {
  static const int rad[] = {2, 3, 4, 5, 6, 7, 8, 9, 10, 12, 14, 15, 16};
  auto is = [&](int m, int most) {
    for (int a : rad)
      if (a == m) return m <= most;
    return false;
  };
  if (is(n, last)) {
    *ns = 1;
    r[0] = n;
    return true;
  }
  for (int a : rad)
    if (n % a == 0 && is(n / a, std::min(a, last))) {
      *ns = 2;
      r[0] = a;
      r[1] = n / a;
      return true;
    }
  for (int a : rad)
    for (int b : rad)
      if (b <= a && n % (a * b) == 0 && is(n / (a * b), std::min(b, last))) {
        *ns = 3;
        r[0] = a;
        r[1] = b;
        r[2] = n / (a * b);
        return true;
      }
  return false;
}

// Columns per block: 128 bytes of a row (16 FP32, 8 FP64), fewer where the
// buffer (two for three stages) and the tables would pass 64 KB.  Threads
// for one butterfly each of the smaller radix, at most 16 x 16, so that a
// two-stage convolution exchanges within one buffer.
static void column_plan(int n, int ncol, size_t csz, size_t tsz, bool conv,
                        ColPlan *p) {
  *p = ColPlan{};
  if (!fft_radices(n, 16, &p->ns, p->r)) return;
  const int nbuf = p->ns == 3 ? 2 : 1;
  const size_t tab = (size_t)n * tsz + (conv ? 2 * (size_t)(n / 2 + 1) * sizeof(double) : 0);
  int lgT = csz == 8 ? 4 : 3;
  while (lgT > 0 && tab + ((nbuf * (size_t)n * csz) << lgT) > kColLds) --lgT;
  const size_t lds = tab + ((nbuf * (size_t)n * csz) << lgT);
  if (lds > kColLds) {
    p->ns = 0;
    return;
  }
  p->n = n;
  p->lgT = lgT;
  p->ncol = ncol;
  p->nblk = (ncol + (1 << lgT) - 1) >> lgT;
  const int items = (n / p->r[p->ns - 1]) << lgT;
  p->nthr = std::min(256, std::max(64, (items + 63) / 64 * 64));
  p->lds = (int)lds;
}

void column_plans(int prec, const int s[3], ColPlan *cy, ColPlan *cz) {
  const bool f = prec == MFE_PREC_MIXED;
  const size_t csz = f ? sizeof(cplx<float>) : sizeof(cplx<double>);
  const size_t tsz = f ? sizeof(Twiddle<float>) : sizeof(Twiddle<double>);
  const int hx = s[0] / 2 + 1;
  column_plan(s[1], s[2] * hx, csz, tsz, false, cy);
  column_plan(s[2], s[1] * hx, csz, tsz, true, cz);
}

void fft_y(const Group &g, int inverse) {
#define MFE_Y(T)                                                                              \
  do {                                                                                        \
    const dim3 gc(g.cy_blocks, 1, g.R), gr(g.fy_x, g.fy_y, g.R);                              \
    if (g.cy_blocks && inverse)                                                               \
      hipLaunchKernelGGL((k_col_y<T, true>), gc, dim3(g.cy_thr), g.lds_cy, g.stream, g.d);    \
    else if (g.cy_blocks)                                                                     \
      hipLaunchKernelGGL((k_col_y<T, false>), gc, dim3(g.cy_thr), g.lds_cy, g.stream, g.d);   \
    if (g.fy_x)                                                                               \
      hipLaunchKernelGGL(k_fft_y<T>, gr, dim3(256), g.lds_fy, g.stream, g.d, inverse);        \
  } while (0)
  if (g.prec == MFE_PREC_MIXED) MFE_Y(float);
  else MFE_Y(double);
#undef MFE_Y
}
void fft_z_forward(const Group &g, void *out) {
#define MFE_Z(T)                                                                              \
  do {                                                                                        \
    const dim3 gc(g.cz_blocks, 1, g.R), gr(g.fz_x, g.fz_y, g.R);                              \
    if (g.cz_blocks)                                                                          \
      hipLaunchKernelGGL(k_col_z_fwd<T>, gc, dim3(g.cz_thr), g.lds_cz, g.stream, g.d, out);   \
    if (g.fz_x)                                                                               \
      hipLaunchKernelGGL(k_fft_z_fwd<T>, gr, dim3(256), g.lds_fz, g.stream, g.d, out);        \
  } while (0)
  if (g.prec == MFE_PREC_MIXED) MFE_Z(float);
  else MFE_Z(double);
#undef MFE_Z
}
void fft_conv(const Group &g, bool energy) {
#define MFE_C(T)                                                                              \
  do {                                                                                        \
    const dim3 gc(g.cz_blocks, 1, g.R), gr(g.fz_x, g.fz_y, g.R);                              \
    const int en = energy ? 1 : 0;                                                            \
    if (g.cz_blocks)                                                                          \
      hipLaunchKernelGGL(k_col_conv<T>, gc, dim3(g.cz_thr), g.lds_cz, g.stream, g.d, en);     \
    if (g.fz_x)                                                                               \
      hipLaunchKernelGGL(k_fft_conv<T>, gr, dim3(256), g.lds_fz, g.stream, g.d, en);          \
  } while (0)
  if (g.prec == MFE_PREC_MIXED) MFE_C(float);
  else MFE_C(double);
#undef MFE_C
}

}  // namespace mfe

