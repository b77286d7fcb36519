// mfe_fft_device.h -- device building blocks of the 3D FFT of SPMFFTRec
// (Src/energy.F90:6525-6587): complex arithmetic with compensated FP32
// twiddles, the LDS-staged mixed-radix Stockham transform, and the passes
// over one block's rows or tiles of one replica's mesh.  The pass kernels
// (mfe_fft.hip, mfe_fft_rows.hip) run one pass over many blocks; the persistent batched step
// (mfe_kernels.hip) runs all passes of a replica in one workgroup.
#pragma once

#include <hip/hip_runtime.h>

#include <type_traits>
#include <utility>

#include "mfe_internal.h"

namespace mfe {
namespace {

template <typename R>
__device__ __forceinline__ cplx<R> cadd(cplx<R> a, cplx<R> b) {
  return {a.x + b.x, a.y + b.y};
}
template <typename R>
__device__ __forceinline__ cplx<R> csub(cplx<R> a, cplx<R> b) {
  return {a.x - b.x, a.y - b.y};
}
template <typename R>
__device__ __forceinline__ cplx<R> conjc(cplx<R> a) {
  return {a.x, -a.y};
}

// v * w (v * conj(w) with cj, the inverse transforms).  FP32 forward: the
// twiddle's residual enters the products through FMA, so the result is the
// product with the exact twiddle, rounded, and carries no magnitude bias
// (the reciprocal energy is a sum of squared forward outputs).  The inverse
// transforms feed only the forces, whose tolerance is far above that bias.
__device__ __forceinline__ cplx<float> twmul(cplx<float> v, const Twiddle<float> &w, bool cj) {
  if (cj) return {v.x * w.x + v.y * w.y, v.y * w.x - v.x * w.y};
  const float c1 = v.x * w.lx - v.y * w.ly, c2 = v.x * w.ly + v.y * w.lx;
  return {__builtin_fmaf(v.x, w.x, __builtin_fmaf(-v.y, w.y, c1)),
          __builtin_fmaf(v.x, w.y, __builtin_fmaf(v.y, w.x, c2))};
}
__device__ __forceinline__ cplx<double> twmul(cplx<double> v, const Twiddle<double> &w,
                                              bool cj) {
  const double wy = cj ? -w.y : w.y;
  return {v.x * w.x - v.y * wy, v.x * wy + v.y * w.x};
}

// x * sqrt(1/2): FP32 forward with the constant's rounding residual added
// by FMA (RN(sqrt(1/2)) is below sqrt(1/2))
__device__ __forceinline__ float mul_sqrt_half(float x, bool inv) {
  return inv ? x * 0.70710677f : __builtin_fmaf(x, 0.70710677f, x * 1.2101617e-08f);
}
__device__ __forceinline__ double mul_sqrt_half(double x, bool) {
  return x * 0.70710678118654752440;
}

constexpr int kMaxRadix = 32;

// e = threadIdx.x + k blockDim.x < n in batches of 8 per thread: the global
// loads of a batch are all issued before the first is stored to LDS, so a
// thread waits for one load latency per batch instead of per element
template <typename Load, typename Store>
__device__ __forceinline__ void batched_copy(int n, Load load, Store store) {
  constexpr int kU = 8;
  for (int e0 = threadIdx.x; e0 < n; e0 += kU * blockDim.x) {
    decltype(load(0)) v[kU];
#pragma unroll
    for (int u = 0; u < kU; ++u) {
      const int e = e0 + u * blockDim.x;
      if (e < n) v[u] = load(e);
    }
#pragma unroll
    for (int u = 0; u < kU; ++u) {
      const int e = e0 + u * blockDim.x;
      if (e < n) store(e, v[u]);
    }
  }
}

// a twiddle table of n entries copied to LDS (read by every stage)
template <typename R>
__device__ __forceinline__ void stage_twiddles(Twiddle<R> *dst,
                                               const Twiddle<R> *__restrict__ src, int n) {
  for (int k = threadIdx.x; k < n; k += blockDim.x) dst[k] = src[k];
}

// R-point DFT of v[0..RAD-1] in registers: V[q] = sum_j v[j] w^(j q), with
// w = exp(-+2 pi i / RAD) taken from the length-n table tw (RAD divides n).
template <typename R, int RAD>
__device__ __forceinline__ void small_dft(cplx<R> *v, bool inv,
                                          const Twiddle<R> *tw, int n) {
  if constexpr (RAD == 2) {
    cplx<R> a = v[0], b = v[1];
    v[0] = cadd(a, b);
    v[1] = csub(a, b);
  } else if constexpr (RAD == 4) {
    cplx<R> a = v[0], b = v[1], c = v[2], d = v[3];
    cplx<R> s0 = cadd(a, c), s1 = csub(a, c), s2 = cadd(b, d), s3 = csub(b, d);
    // forward: -i * s3 ; inverse: +i * s3
    cplx<R> js3 = inv ? cplx<R>{-s3.y, s3.x} : cplx<R>{s3.y, -s3.x};
    v[0] = cadd(s0, s2);
    v[2] = csub(s0, s2);
    v[1] = cadd(s1, js3);
    v[3] = csub(s1, js3);
  } else if constexpr (RAD == 8) {
    // radix 2 x 4: two 4-point DFTs of the even and odd samples, then the
    // odd half twiddled by w8^q (w8 = e^{-+i pi/4})
    cplx<R> e[4] = {v[0], v[2], v[4], v[6]}, o[4] = {v[1], v[3], v[5], v[7]};
    small_dft<R, 4>(e, inv, tw, n);
    small_dft<R, 4>(o, inv, tw, n);
    // o[1] *= w8, o[2] *= w8^2 = -+i, o[3] *= w8^3
    const R sg = inv ? R(1) : R(-1);
    cplx<R> o1 = {mul_sqrt_half(o[1].x - sg * o[1].y, inv),
                  mul_sqrt_half(o[1].y + sg * o[1].x, inv)};
    cplx<R> o2 = {-sg * o[2].y, sg * o[2].x};
    cplx<R> o3 = {mul_sqrt_half(-o[3].x - sg * o[3].y, inv),
                  mul_sqrt_half(-o[3].y + sg * o[3].x, inv)};
    v[0] = cadd(e[0], o[0]);
    v[4] = csub(e[0], o[0]);
    v[1] = cadd(e[1], o1);
    v[5] = csub(e[1], o1);
    v[2] = cadd(e[2], o2);
    v[6] = csub(e[2], o2);
    v[3] = cadd(e[3], o3);
    v[7] = csub(e[3], o3);
  } else {
    cplx<R> out[RAD];
    const int step = n / RAD;
#pragma unroll
    for (int qq = 0; qq < RAD; ++qq) {
      cplx<R> acc = v[0];
#pragma unroll
      for (int j = 1; j < RAD; ++j) acc = cadd(acc, twmul(v[j], tw[((j * qq) % RAD) * step], inv));
      out[qq] = acc;
    }
#pragma unroll
    for (int qq = 0; qq < RAD; ++qq) v[qq] = out[qq];
  }
}

// one Stockham stage of radix RAD over `batch` sequences (Govindaraju et
// al., SC'08): j-th butterfly reads in[j + q*n/RAD], twiddles by
// w^(k q) with k = j mod Ns, and writes out[(j/Ns)*Ns*RAD + k + q*Ns]
// lg_nbf / lg_ns: log2 of n/RAD and of Ns when both are powers of two
// (shifts replace the divisions), -1 otherwise.  k q tstep < n, so the
// twiddle index needs no reduction.
template <typename R, int RAD>
__device__ __forceinline__ void stockham_stage(const cplx<R> *a, cplx<R> *b,
                                               int n, int Ns, int batch,
                                               int ld, const Twiddle<R> *tw,
                                               bool inv, int lg_nbf, int lg_ns) {
  const int nbf = n / RAD;
  const int total = nbf * batch;
  const int tstep = n / (Ns * RAD);
  for (int t = threadIdx.x; t < total; t += blockDim.x) {
    int sq, j, jb, k;
    if (lg_nbf >= 0) {
      sq = t >> lg_nbf;
      j = t & (nbf - 1);
      jb = j >> lg_ns;
      k = j & (Ns - 1);
    } else {
      sq = t / nbf;
      j = t - sq * nbf;
      jb = j / Ns;
      k = j - jb * Ns;
    }
    const cplx<R> *in = a + sq * ld;
    cplx<R> *out = b + sq * ld;
    cplx<R> v[RAD];
#pragma unroll
    for (int q = 0; q < RAD; ++q) v[q] = in[j + q * nbf];
#pragma unroll
    for (int q = 1; q < RAD; ++q) v[q] = twmul(v[q], tw[k * q * tstep], inv);
    small_dft<R, RAD>(v, inv, tw, n);
    const int base = jb * Ns * RAD + k;
#pragma unroll
    for (int q = 0; q < RAD; ++q) out[base + q * Ns] = v[q];
  }
}

// generic prime radix up to kMaxRadix (meshes with large prime factors)
template <typename R>
__device__ __forceinline__ void stockham_stage_generic(const cplx<R> *a, cplx<R> *b, int n,
                                       int Ns, int rad, int batch, int ld,
                                       const Twiddle<R> *tw, bool inv) {
  const int nbf = n / rad;
  const int total = nbf * batch;
  const int tstep = n / (Ns * rad);
  const int step = n / rad;
  for (int t = threadIdx.x; t < total; t += blockDim.x) {
    const int sq = t / nbf, j = t - sq * nbf;
    const cplx<R> *in = a + sq * ld;
    cplx<R> *out = b + sq * ld;
    const int k = j % Ns;
    const int base = (j / Ns) * Ns * rad + k;
    for (int qq = 0; qq < rad; ++qq) {
      cplx<R> acc = {R(0), R(0)};
      for (int q = 0; q < rad; ++q) {
        acc = cadd(acc, twmul(in[j + q * nbf], tw[((k * q * tstep) + ((q * qq) % rad) * step) % n],
                              inv));
      }
      out[base + qq * Ns] = acc;
    }
  }
}

// Batched Stockham FFT staged in LDS: `batch` sequences of length p.n at
// a[s*ld + k]; b is scratch of the same shape.  Returns the buffer holding
// the result in natural order.  All threads of the block take part.
template <typename R>
__device__ __forceinline__ cplx<R> *lds_fft(cplx<R> *a, cplx<R> *b, const FftPlan &p,
                            int batch, int ld, const Twiddle<R> *tw, bool inv) {
  const int n = p.n;
  int Ns = 1;
  const bool pow2 = (n & (n - 1)) == 0;
  for (int st = 0; st < p.nstages; ++st) {
    const int r = p.radix[st];
    const int lg_nbf = pow2 ? __builtin_ctz(n / r) : -1;
    const int lg_ns = pow2 ? __builtin_ctz(Ns) : -1;
    switch (r) {
      case 8: stockham_stage<R, 8>(a, b, n, Ns, batch, ld, tw, inv, lg_nbf, lg_ns); break;
      case 4: stockham_stage<R, 4>(a, b, n, Ns, batch, ld, tw, inv, lg_nbf, lg_ns); break;
      case 2: stockham_stage<R, 2>(a, b, n, Ns, batch, ld, tw, inv, lg_nbf, lg_ns); break;
      case 3: stockham_stage<R, 3>(a, b, n, Ns, batch, ld, tw, inv, lg_nbf, lg_ns); break;
      case 5: stockham_stage<R, 5>(a, b, n, Ns, batch, ld, tw, inv, lg_nbf, lg_ns); break;
      case 7: stockham_stage<R, 7>(a, b, n, Ns, batch, ld, tw, inv, lg_nbf, lg_ns); break;
      default: stockham_stage_generic<R>(a, b, n, Ns, r, batch, ld, tw, inv); break;
    }
    __syncthreads();
    cplx<R> *tmp = a;
    a = b;
    b = tmp;
    Ns *= r;
  }
  return a;
}

// ------------------------------------------------ transforms in registers
// The column passes (y and z) transform a length n = r1 r2 (r3) of radices
// up to 16 with one radix per stage held in a thread's registers: the first
// stage reads global memory, the last writes it, and only the one or two
// exchanges between go through LDS.  A Stockham transform staged through
// LDS on both ends (lds_fft) moves every value through LDS once more per
// end and waits at twice as many barriers: 128 points in three stages took
// eight LDS passes and five barriers, 16 x 8 in registers takes two and one.

// cos and sin of 2 pi k / n, reduced to the first octant (Taylor series)
struct Trig {
  double c, s;
};
constexpr Trig trig_root(int k, int n) {
  k %= n;
  if (2 * k > n) {
    const Trig t = trig_root(n - k, n);
    return {t.c, -t.s};
  }
  if (4 * k > n) {
    const Trig t = trig_root(n - 2 * k, 2 * n);
    return {-t.c, t.s};
  }
  if (8 * k > n) {
    const Trig t = trig_root(n - 4 * k, 4 * n);
    return {t.s, t.c};
  }
  const double x = 6.283185307179586476925286766559 * k / n;
  double c = 0.0, s = 0.0;
  // Horner from x^21 and x^20 down: below 1e-20 of the sum for x <= pi/4
  for (int j = 10; j >= 0; --j) {
    s = 1.0 - s * x * x / ((2 * j + 2) * (2 * j + 3));
    c = 1.0 - c * x * x / ((2 * j + 1) * (2 * j + 2));
  }
  return {c, s * x};
}

template <int N, typename F, int... I>
__device__ __forceinline__ void static_for_impl(F &&f, std::integer_sequence<int, I...>) {
  (f(std::integral_constant<int, I>{}), ...);
}
template <int N, typename F>
__device__ __forceinline__ void static_for(F &&f) {
  static_for_impl<N>(f, std::make_integer_sequence<int, N>{});
}

// acc + x * C for a constant C; FP32 forward with the constant's rounding
// residual added by FMA (see Twiddle)
template <typename R, bool INV>
__device__ __forceinline__ R mac_const(R acc, R x, double c) {
  if constexpr (sizeof(R) == 4) {
    const float hi = (float)c;
    if constexpr (INV) return __builtin_fmaf(x, hi, acc);
    return __builtin_fmaf(x, hi, __builtin_fmaf(x, (float)(c - (double)hi), acc));
  } else {
    return __builtin_fma(x, c, acc);
  }
}

// v * exp(-2 pi i K / N) (forward) or its conjugate (inverse)
template <typename R, int K, int N, bool INV>
__device__ __forceinline__ cplx<R> mul_root(cplx<R> v) {
  constexpr int k = K % N;
  constexpr R sg = INV ? R(1) : R(-1);  // w = c + i sg s
  if constexpr (k == 0) {
    return v;
  } else if constexpr (4 * k == N) {
    return {-sg * v.y, sg * v.x};
  } else if constexpr (2 * k == N) {
    return {-v.x, -v.y};
  } else if constexpr (4 * k == 3 * N) {
    return {sg * v.y, -sg * v.x};
  } else {
    constexpr Trig t = trig_root(k, N);
    constexpr double s = INV ? t.s : -t.s;
    return {mac_const<R, INV>(mac_const<R, INV>(R(0), v.x, t.c), v.y, -s),
            mac_const<R, INV>(mac_const<R, INV>(R(0), v.y, t.c), v.x, s)};
  }
}

// RAD-point DFT in registers, natural order in and out
template <typename R, int RAD, bool INV>
__device__ __forceinline__ void reg_dft(cplx<R> *v) {
  if constexpr (RAD == 2 || RAD == 4 || RAD == 8) {
    small_dft<R, RAD>(v, INV, nullptr, 0);
  } else if constexpr (RAD == 3 || RAD == 5 || RAD == 7) {
    constexpr int H = (RAD - 1) / 2;
    cplx<R> t[H], u[H];
#pragma unroll
    for (int j = 0; j < H; ++j) {
      t[j] = cadd(v[j + 1], v[RAD - 1 - j]);
      u[j] = csub(v[j + 1], v[RAD - 1 - j]);
    }
    const cplx<R> v0 = v[0];
#pragma unroll
    for (int j = 0; j < H; ++j) v[0] = cadd(v[0], t[j]);
    static_for<H>([&](auto qi) {
      constexpr int q = decltype(qi)::value + 1;
      cplx<R> a = v0, b = {R(0), R(0)};
      static_for<H>([&](auto ji) {
        constexpr int j = decltype(ji)::value + 1;
        constexpr Trig w = trig_root(j * q, RAD);
        a.x = mac_const<R, INV>(a.x, t[j - 1].x, w.c);
        a.y = mac_const<R, INV>(a.y, t[j - 1].y, w.c);
        b.x = mac_const<R, INV>(b.x, u[j - 1].x, w.s);
        b.y = mac_const<R, INV>(b.y, u[j - 1].y, w.s);
      });
      // a -+ i b
      const cplx<R> ib = INV ? cplx<R>{-b.y, b.x} : cplx<R>{b.y, -b.x};
      v[q] = cadd(a, ib);
      v[RAD - q] = csub(a, ib);
    });
  } else {
    // A x B: A-point DFTs over stride B, the roots of RAD, B-point DFTs
    constexpr int A = RAD % 7 == 0 ? 7 : (RAD % 5 == 0 ? 5 : (RAD == 12 || RAD == 16 ? 4 : 3));
    constexpr int B = RAD / A;
    static_assert(A * B == RAD, "radix of two factors");
    cplx<R> y[RAD];  // y[k1 B + n2]
    static_for<B>([&](auto n2i) {
      constexpr int n2 = decltype(n2i)::value;
      cplx<R> x[A];
#pragma unroll
      for (int n1 = 0; n1 < A; ++n1) x[n1] = v[n1 * B + n2];
      reg_dft<R, A, INV>(x);
      static_for<A>([&](auto k1i) {
        constexpr int k1 = decltype(k1i)::value;
        y[k1 * B + n2] = mul_root<R, k1 * n2, RAD, INV>(x[k1]);
      });
    });
#pragma unroll
    for (int k1 = 0; k1 < A; ++k1) {
      reg_dft<R, B, INV>(y + k1 * B);
#pragma unroll
      for (int k2 = 0; k2 < B; ++k2) v[k1 + A * k2] = y[k1 * B + k2];
    }
  }
}

// One stage of radix RAD for T = 1 << lgT columns of length n, Ns points
// already combined: butterfly j of column c reads positions j + q n/RAD,
// multiplies by w_{Ns RAD}^{q (j mod Ns)}, transforms and writes positions
// (j / Ns) Ns RAD + j mod Ns + q Ns.  POS: first stage (Ns 1, no twiddles),
// middle, last (Ns RAD = n, so j < Ns).  rd(pos, c), wr(pos, c, v).
enum { ST_FIRST = 0, ST_MID = 1, ST_LAST = 2 };
template <typename R, int RAD, bool INV, int POS>
__device__ __forceinline__ void stage_twiddle(cplx<R> *v, int j, int n, int Ns, int &base,
                                              const Twiddle<R> *tw) {
  if constexpr (POS == ST_FIRST) {
    base = j * RAD;
  } else {
    const int jb = POS == ST_LAST ? 0 : j / Ns, k = j - jb * Ns;
    const int kt = POS == ST_LAST ? k : k * (n / (Ns * RAD));
#pragma unroll
    for (int q = 1; q < RAD; ++q) v[q] = twmul(v[q], tw[kt * q], INV);
    base = jb * Ns * RAD + k;
  }
}
template <typename R, int RAD, bool INV, int POS, typename Rd, typename Wr>
__device__ __forceinline__ void col_stage(int n, int lgT, int nt, int Ns, const Twiddle<R> *tw,
                                          Rd rd, Wr wr) {
  const int nb = n / RAD, step = POS == ST_FIRST ? 1 : Ns;
  for (int t = threadIdx.x; t < nb << lgT; t += blockDim.x) {
    const int c = t & ((1 << lgT) - 1), j = t >> lgT;
    if (c >= nt) continue;
    cplx<R> v[RAD];
#pragma unroll
    for (int q = 0; q < RAD; ++q) v[q] = rd(j + q * nb, c);
    int base;
    stage_twiddle<R, RAD, INV, POS>(v, j, n, Ns, base, tw);
    reg_dft<R, RAD, INV>(v);
#pragma unroll
    for (int q = 0; q < RAD; ++q) wr(base + q * step, c, v[q]);
  }
}

#define MFE_FOR_RADIX(r, CALL) \
  switch (r) {                 \
    case 2: CALL(2); break;    \
    case 3: CALL(3); break;    \
    case 4: CALL(4); break;    \
    case 5: CALL(5); break;    \
    case 6: CALL(6); break;    \
    case 7: CALL(7); break;    \
    case 8: CALL(8); break;    \
    case 9: CALL(9); break;    \
    case 10: CALL(10); break;  \
    case 12: CALL(12); break;  \
    case 14: CALL(14); break;  \
    case 15: CALL(15); break;  \
    default: CALL(16); break;  \
  }

template <typename R, bool INV, int POS, typename Rd, typename Wr>
__device__ __forceinline__ void any_stage(int rad, int n, int lgT, int nt, int Ns,
                                          const Twiddle<R> *tw, Rd rd, Wr wr) {
#define MFE_CALL(RAD) col_stage<R, RAD, INV, POS>(n, lgT, nt, Ns, tw, rd, wr)
  MFE_FOR_RADIX(rad, MFE_CALL)
#undef MFE_CALL
}

// The transform of one block's columns: rd(pos, c) reads the input, wr
// writes the output; A and B hold T n values each (B only for three stages).
// tw: the length-n twiddles (in LDS: staged by the caller before, read
// after the first barrier).
template <typename R, bool INV, typename Rd, typename Wr>
__device__ __forceinline__ void col_fft(const ColPlan &p, int nt, cplx<R> *A, cplx<R> *B,
                                        const Twiddle<R> *tw, Rd rd, Wr wr) {
  const int n = p.n, lgT = p.lgT;
  auto put = [&](cplx<R> *buf) {
    return [=](int pos, int c, cplx<R> v) { buf[(pos << lgT) + c] = v; };
  };
  auto get = [&](const cplx<R> *buf) {
    return [=](int pos, int c) { return buf[(pos << lgT) + c]; };
  };
  if (p.ns == 1) {
    any_stage<R, INV, ST_FIRST>(p.r[0], n, lgT, nt, 1, tw, rd, wr);
    return;
  }
  any_stage<R, INV, ST_FIRST>(p.r[0], n, lgT, nt, 1, tw, rd, put(A));
  __syncthreads();
  if (p.ns == 2) {
    any_stage<R, INV, ST_LAST>(p.r[1], n, lgT, nt, p.r[0], tw, get(A), wr);
    return;
  }
  any_stage<R, INV, ST_MID>(p.r[1], n, lgT, nt, p.r[0], tw, get(A), put(B));
  __syncthreads();
  any_stage<R, INV, ST_LAST>(p.r[2], n, lgT, nt, p.r[0] * p.r[1], tw, get(B), wr);
}

// The forward transform's last stage, f(pos, c, v) applied to each output,
// and the inverse transform's first stage (the radices in reverse order) in
// the same registers: the outputs j + q n/RAD of one are the inputs of the
// other.
// ONE: rd and wr share a buffer; every thread has at most one butterfly and
// all have read before any writes.
template <typename R, int RAD, bool ONE, typename Rd, typename Fn, typename Wr>
__device__ __forceinline__ void conv_stage(int n, int lgT, int nt, const Twiddle<R> *tw, Rd rd,
                                           Fn f, Wr wr) {
  const int nb = n / RAD, items = nb << lgT;
  const int t_end = ONE ? (int)threadIdx.x + 1 : items;
  for (int t = threadIdx.x; t < t_end; t += blockDim.x) {
    const int c = t & ((1 << lgT) - 1), j = t >> lgT;
    const bool act = t < items && c < nt;
    cplx<R> v[RAD];
    if (act) {
#pragma unroll
      for (int q = 0; q < RAD; ++q) v[q] = rd(j + q * nb, c);
    }
    if (ONE) __syncthreads();
    if (!act) continue;
    if (nb > 1) {
#pragma unroll
      for (int q = 1; q < RAD; ++q) v[q] = twmul(v[q], tw[j * q], false);
    }
    reg_dft<R, RAD, false>(v);
#pragma unroll
    for (int q = 0; q < RAD; ++q) v[q] = f(j + q * nb, c, v[q]);
    reg_dft<R, RAD, true>(v);
#pragma unroll
    for (int q = 0; q < RAD; ++q) wr(j * RAD + q, c, v[q]);
  }
}
template <typename R, bool ONE, typename Rd, typename Fn, typename Wr>
__device__ __forceinline__ void any_conv_stage(int rad, int n, int lgT, int nt,
                                               const Twiddle<R> *tw, Rd rd, Fn f, Wr wr) {
#define MFE_CALL(RAD) conv_stage<R, RAD, ONE>(n, lgT, nt, tw, rd, f, wr)
  MFE_FOR_RADIX(rad, MFE_CALL)
#undef MFE_CALL
}

// forward transform, f on every element, inverse transform, of one block's
// columns
template <typename R, typename Rd, typename Fn, typename Wr>
__device__ __forceinline__ void col_conv(const ColPlan &p, int nt, cplx<R> *A, cplx<R> *B,
                                         const Twiddle<R> *tw, Rd rd, Fn f, Wr wr) {
  const int n = p.n, lgT = p.lgT;
  auto put = [&](cplx<R> *buf) {
    return [=](int pos, int c, cplx<R> v) { buf[(pos << lgT) + c] = v; };
  };
  auto get = [&](const cplx<R> *buf) {
    return [=](int pos, int c) { return buf[(pos << lgT) + c]; };
  };
  if (p.ns == 1) {
    any_conv_stage<R, false>(p.r[0], n, lgT, nt, tw, rd, f, wr);
    return;
  }
  any_stage<R, false, ST_FIRST>(p.r[0], n, lgT, nt, 1, tw, rd, put(A));
  __syncthreads();
  if (p.ns == 2) {
    any_conv_stage<R, true>(p.r[1], n, lgT, nt, tw, get(A), f, put(A));
    __syncthreads();
    any_stage<R, true, ST_LAST>(p.r[0], n, lgT, nt, p.r[1], tw, get(A), wr);
    return;
  }
  any_stage<R, false, ST_MID>(p.r[1], n, lgT, nt, p.r[0], tw, get(A), put(B));
  __syncthreads();
  any_conv_stage<R, false>(p.r[2], n, lgT, nt, tw, get(B), f, put(A));
  __syncthreads();
  any_stage<R, true, ST_MID>(p.r[1], n, lgT, nt, p.r[2], tw, get(A), put(B));
  __syncthreads();
  any_stage<R, true, ST_LAST>(p.r[0], n, lgT, nt, p.r[2] * p.r[1], tw, get(B), wr);
}

// --------------------------------------------------- x rows in registers
// The r2c and c2r transforms of rows of s1 = 2m reals through a complex
// transform of length m (fftx_fwd_rows has the formulas), with the radices
// of col_fft: butterfly j of row c, j fastest over the threads.  The pass
// that combines Z[k] with Z[m-k] takes the butterflies j and Ns - j of the
// forward transform's last stage (the inverse's first) in one thread, whose
// outputs (inputs) j + q Ns and m - (j + q Ns) then pair up in registers.
// Both ends of that pair of stages take the plan's smallest radix, at most
// 8 (two butterflies are held at once); the inverse runs the radices in
// reverse order.
//
// Outputs of butterfly j (nb butterflies in all) are Z[j + q nb]; with j2 = nb - j the partner of
// element q is element RAD-1-q of the sequence j2 + i nb.  For j = 0 that
// sequence is nb, 2 nb, ..., m (Z[m] = Z[0]).
#define MFE_FOR_RADIX8(r, CALL) \
  switch (r) {                  \
    case 2: CALL(2); break;     \
    case 3: CALL(3); break;     \
    case 4: CALL(4); break;     \
    case 5: CALL(5); break;     \
    case 6: CALL(6); break;     \
    case 7: CALL(7); break;     \
    default: CALL(8); break;    \
  }
template <typename R, int RAD>
__device__ __forceinline__ void r2c_stage(const RowPlan &p, int nr, const Twiddle<R> *twh,
                                          const Twiddle<R> *twf, const cplx<R> *in,
                                          cplx<R> *__restrict__ out) {
  const int m = p.m, nb = m / RAD, np = nb / 2 + 1, hx = m + 1;
  for (int t = threadIdx.x; t < nr * np; t += blockDim.x) {
    const int c = fdiv(t, p.f_pair), j = t - c * np;
    const bool self = j == 0 || 2 * j == nb;
    const cplx<R> *row = in + c * p.ld;
    cplx<R> v[RAD], u[RAD];
    auto butterfly = [&](cplx<R> *w, int jj) {
#pragma unroll
      for (int q = 0; q < RAD; ++q) w[q] = row[jj + q * nb];
      if (nb > 1) {
#pragma unroll
        for (int q = 1; q < RAD; ++q) w[q] = twmul(w[q], twh[jj * q], false);
      }
      reg_dft<R, RAD, false>(w);
    };
    butterfly(v, j);
    if (!self) {
      butterfly(u, nb - j);
    } else {
#pragma unroll
      for (int q = 0; q < RAD; ++q) u[q] = j == 0 ? v[(q + 1) % RAD] : v[q];
    }
    cplx<R> *orow = out + (size_t)c * hx;
    auto put = [&](cplx<R> zk, cplx<R> zmk, int k) {
      const cplx<R> zm = conjc(zmk);
      const cplx<R> ev = {(zk.x + zm.x) * R(0.5), (zk.y + zm.y) * R(0.5)};
      const cplx<R> d = csub(zk, zm);
      const cplx<R> od = {d.y * R(0.5), -d.x * R(0.5)};
      orow[k] = cadd(ev, twmul(od, twf[k], false));
    };
#pragma unroll
    for (int q = 0; q < RAD; ++q) put(v[q], u[RAD - 1 - q], j + q * nb);
    if (!self) {
#pragma unroll
      for (int q = 0; q < RAD; ++q) put(u[q], v[RAD - 1 - q], nb - j + q * nb);
    }
    if (j == 0) put(v[0], v[0], m);
  }
}

// the inverse's first stage: X of a row from global memory, Z and its
// butterflies j and nb - j, written to positions j RAD + q by wr(pos, c, v)
template <typename R, int RAD, typename Wr>
__device__ __forceinline__ void c2r_stage(const RowPlan &p, int nr, const Twiddle<R> *twf,
                                          const cplx<R> *__restrict__ in, Wr wr) {
  const int m = p.m, nb = m / RAD, np = nb / 2 + 1, hx = m + 1;
  for (int t = threadIdx.x; t < nr * np; t += blockDim.x) {
    const int c = fdiv(t, p.f_pair), j = t - c * np;
    const bool self = j == 0 || 2 * j == nb;
    const cplx<R> *row = in + (size_t)c * hx;
    cplx<R> x[RAD], y[RAD];
#pragma unroll
    for (int q = 0; q < RAD; ++q) {
      x[q] = row[j + q * nb];
      y[q] = row[nb - j + q * nb];
    }
    if (j == 0) {
      // Re(X[0]) and Re(X[m]) only
      x[0].y = R(0);
      y[RAD - 1].y = R(0);
    }
    auto pre = [&](cplx<R> xk, cplx<R> xmk, int k) -> cplx<R> {
      const cplx<R> xm = conjc(xmk);
      const cplx<R> A = cadd(xk, xm), D = csub(xk, xm);
      const cplx<R> Dw = twmul(D, twf[k], true);
      return {A.x - Dw.y, A.y + Dw.x};
    };
    cplx<R> z[RAD];
#pragma unroll
    for (int q = 0; q < RAD; ++q) z[q] = pre(x[q], y[RAD - 1 - q], j + q * nb);
    reg_dft<R, RAD, true>(z);
#pragma unroll
    for (int q = 0; q < RAD; ++q) wr(j * RAD + q, c, z[q]);
    if (!self) {
#pragma unroll
      for (int q = 0; q < RAD; ++q) z[q] = pre(y[q], x[RAD - 1 - q], nb - j + q * nb);
      reg_dft<R, RAD, true>(z);
#pragma unroll
      for (int q = 0; q < RAD; ++q) wr((nb - j) * RAD + q, c, z[q]);
    }
  }
}

// a plain stage of the rows: as col_stage with j fastest (st: the stage's
// place in the plan, whose butterflies per row are p.f_nb[st].d)
template <typename R, int RAD, bool INV, int POS, typename Rd, typename Wr>
__device__ __forceinline__ void row_stage(const RowPlan &p, int nr, int st, int Ns,
                                          const Twiddle<R> *tw, Rd rd, Wr wr) {
  const int n = p.m, nb = n / RAD, step = POS == ST_FIRST ? 1 : Ns;
  for (int t = threadIdx.x; t < nr * nb; t += blockDim.x) {
    const int c = fdiv(t, p.f_nb[st]), j = t - c * nb;
    cplx<R> v[RAD];
#pragma unroll
    for (int q = 0; q < RAD; ++q) v[q] = rd(j + q * nb, c);
    int base;
    stage_twiddle<R, RAD, INV, POS>(v, j, n, Ns, base, tw);
    reg_dft<R, RAD, INV>(v);
#pragma unroll
    for (int q = 0; q < RAD; ++q) wr(base + q * step, c, v[q]);
  }
}
template <typename R, bool INV, int POS, typename Rd, typename Wr>
__device__ __forceinline__ void any_row_stage(const RowPlan &p, int nr, int st, int Ns,
                                              const Twiddle<R> *tw, Rd rd, Wr wr) {
#define MFE_CALL(RAD) row_stage<R, RAD, INV, POS>(p, nr, st, Ns, tw, rd, wr)
  MFE_FOR_RADIX(p.r[st], MFE_CALL)
#undef MFE_CALL
}

// forward: nr rows of reals in A (row c at 2 c ld), transformed into out
// ([nr][m + 1]); B a second buffer of the same size
template <typename R>
__device__ __forceinline__ void rows_fwd(const RowPlan &p, int nr, cplx<R> *A, cplx<R> *B,
                                         const Twiddle<R> *twh, const Twiddle<R> *twf,
                                         cplx<R> *__restrict__ out) {
  const int ld = p.ld;
  auto get = [=](const cplx<R> *b) { return [=](int pos, int c) { return b[c * ld + pos]; }; };
  auto put = [=](cplx<R> *b) {
    return [=](int pos, int c, cplx<R> v) { b[c * ld + pos] = v; };
  };
  int Ns = 1;
  if (p.ns >= 2) {
    any_row_stage<R, false, ST_FIRST>(p, nr, 0, 1, twh, get(A), put(B));
    __syncthreads();
    cplx<R> *x = A;
    A = B;
    B = x;
    Ns = p.r[0];
  }
  if (p.ns == 3) {
    any_row_stage<R, false, ST_MID>(p, nr, 1, Ns, twh, get(A), put(B));
    __syncthreads();
    A = B;
  }
#define MFE_CALL(RAD) r2c_stage<R, RAD>(p, nr, twh, twf, A, out)
  MFE_FOR_RADIX8(p.r[p.ns - 1], MFE_CALL)
#undef MFE_CALL
}

// inverse: nr rows of in ([nr][m + 1]) into reals, written as pairs by
// wr(k, c, {x[2k], x[2k+1]})
template <typename R, typename Wr>
__device__ __forceinline__ void rows_inv(const RowPlan &p, int nr, cplx<R> *A, cplx<R> *B,
                                         const Twiddle<R> *twh, const Twiddle<R> *twf,
                                         const cplx<R> *__restrict__ in, Wr wr) {
  const int ld = p.ld;
  auto get = [=](const cplx<R> *b) { return [=](int pos, int c) { return b[c * ld + pos]; }; };
  auto put = [=](cplx<R> *b) {
    return [=](int pos, int c, cplx<R> v) { b[c * ld + pos] = v; };
  };
  if (p.ns == 1) {
#define MFE_CALL(RAD) c2r_stage<R, RAD>(p, nr, twf, in, wr)
    MFE_FOR_RADIX8(p.r[0], MFE_CALL)
#undef MFE_CALL
    return;
  }
#define MFE_CALL(RAD) c2r_stage<R, RAD>(p, nr, twf, in, put(A))
  MFE_FOR_RADIX8(p.r[p.ns - 1], MFE_CALL)
#undef MFE_CALL
  __syncthreads();
  int Ns = p.r[p.ns - 1];
  if (p.ns == 3) {
    any_row_stage<R, true, ST_MID>(p, nr, 1, Ns, twh, get(A), put(B));
    __syncthreads();
    A = B;
    Ns *= p.r[1];
  }
  any_row_stage<R, true, ST_LAST>(p, nr, 0, Ns, twh, get(A), wr);
}

// ----------------------------------------------------------------- x pass
// r2c of rows of length s1 = 2m: z[k] = x[2k] + i x[2k+1], Z = FFT_m(z),
// X[k] = (Z[k] + conj(Z[m-k]))/2 - i/2 (Z[k] - conj(Z[m-k])) W^k.
// Rows blk * fx_rpb, ... of the mesh; load(x, y, z) gives the real mesh
// value at a point.
// rows row0 .. row0 + nr - 1 (nr <= cap, the LDS buffers' row capacity)
template <typename R, typename Load>
__device__ __forceinline__ void fftx_fwd_rows(const SysDev &V, int row0, int nr, int cap,
                                              char *smem, Load load) {
  cplx<R> *__restrict__ cm = (cplx<R> *)V.mesh_c;
  const int s1 = V.sg.s[0], rows_per_blk = cap;
  const FftPlan &ph = V.plan_half;
  const Twiddle<R> *__restrict__ tw_half = (const Twiddle<R> *)V.tw_half;
  const Twiddle<R> *__restrict__ tw_full = (const Twiddle<R> *)V.tw[0];
  const int m = s1 / 2, hx = m + 1, ld = m + 1;
  cplx<R> *a = reinterpret_cast<cplx<R> *>(smem);
  cplx<R> *b = a + rows_per_blk * ld;
  R *ar = reinterpret_cast<R *>(a);
  const int s2 = V.sg.s[1];
  Twiddle<R> *twh_s = reinterpret_cast<Twiddle<R> *>(b + rows_per_blk * ld), *twf_s = twh_s + m;
  stage_twiddles(twh_s, tw_half, m);
  stage_twiddles(twf_s, tw_full, s1);
  batched_copy(
      nr * s1,
      [&](int e) {
        const int r = fdiv(e, V.f_s1), x = e - r * s1;
        const int row = row0 + r, z = fdiv(row, V.f_s2), y = row - z * s2;
        return load(x, y, z);
      },
      [&](int e, R v) {
        const int r = fdiv(e, V.f_s1), x = e - r * s1;
        ar[2 * (r * ld) + x] = v;
      });
  __syncthreads();
  cplx<R> *z = lds_fft(a, b, ph, nr, ld, twh_s, false);
  for (int e = threadIdx.x; e < nr * hx; e += blockDim.x) {
    const int r = fdiv(e, V.f_hx), k = e - r * hx;
    // k in [0, m]: k mod m and (m - k) mod m without divisions
    cplx<R> zk = z[r * ld + (k == m ? 0 : k)];
    cplx<R> zm = conjc(z[r * ld + (k == 0 ? 0 : m - k)]);
    cplx<R> ev = {(zk.x + zm.x) * R(0.5), (zk.y + zm.y) * R(0.5)};
    cplx<R> d = csub(zk, zm);
    cplx<R> od = {d.y * R(0.5), -d.x * R(0.5)};
    cplx<R> X = cadd(ev, twmul(od, twf_s[k], false));
    cm[(size_t)(row0 + r) * hx + k] = X;
  }
}

// c2r of rows: Re(X[0]), Re(X[m]) only (FFTW's reading of a Hermitian row);
// Z[k] = (X[k] + conj(X[m-k])) + i (X[k] - conj(X[m-k])) W^-k, z = IFFT_m(Z),
// x[2j] = Re z[j], x[2j+1] = Im z[j] (unnormalised), into the real mesh.
template <typename R>
__device__ __forceinline__ void fftx_inv_rows(const SysDev &V, int row0, int nr, int cap,
                                              char *smem) {
  const cplx<R> *__restrict__ cm = (const cplx<R> *)V.mesh_c;
  R *__restrict__ real = (R *)V.mesh_r;
  const int s1 = V.sg.s[0], rows_per_blk = cap;
  const FftPlan &ph = V.plan_half;
  const Twiddle<R> *__restrict__ tw_half = (const Twiddle<R> *)V.tw_half;
  const Twiddle<R> *__restrict__ tw_full = (const Twiddle<R> *)V.tw[0];
  const int m = s1 / 2, hx = m + 1, ld = m + 1;
  cplx<R> *a = reinterpret_cast<cplx<R> *>(smem);
  cplx<R> *b = a + rows_per_blk * ld;
  Twiddle<R> *twh_s = reinterpret_cast<Twiddle<R> *>(b + rows_per_blk * ld), *twf_s = twh_s + m;
  stage_twiddles(twh_s, tw_half, m);
  stage_twiddles(twf_s, tw_full, s1);
  batched_copy(
      nr * hx, [&](int e) { return cm[(size_t)row0 * hx + e]; },
      [&](int e, cplx<R> v) {
        const int r = fdiv(e, V.f_hx), k = e - r * hx;
        if (k == 0 || k == m) v.y = R(0);
        b[r * ld + k] = v;
      });
  __syncthreads();
  for (int e = threadIdx.x; e < nr * m; e += blockDim.x) {
    const int r = fdiv(e, V.f_m), k = e - r * m;
    cplx<R> xk = b[r * ld + k];
    cplx<R> xm = conjc(b[r * ld + (m - k)]);
    cplx<R> A = cadd(xk, xm), D = csub(xk, xm);
    cplx<R> Dw = twmul(D, twf_s[k], true);
    a[r * ld + k] = {A.x - Dw.y, A.y + Dw.x};
  }
  __syncthreads();
  cplx<R> *z = lds_fft(a, b, ph, nr, ld, twh_s, true);
  for (int e = threadIdx.x; e < nr * s1; e += blockDim.x) {
    const int r = fdiv(e, V.f_s1), x = e - r * s1;
    cplx<R> v = z[r * ld + (x >> 1)];
    real[(size_t)(row0 + r) * s1 + x] = (x & 1) ? v.y : v.x;
  }
}

// ----------------------------------------------------------------- y pass
// complex FFT along y of kx columns bx * fy_T, ... of plane z
template <typename R>
__device__ __forceinline__ void ffty_tile(const SysDev &V, int bx, int z, int inv, char *smem) {
  cplx<R> *__restrict__ cm = (cplx<R> *)V.mesh_c;
  const int s2 = V.sg.s[1], hx = V.hx, T = V.fy_T;
  const FftPlan &py = V.plan[1];
  const Twiddle<R> *__restrict__ tw = (const Twiddle<R> *)V.tw[1];
  const int ld = s2 + 1;
  cplx<R> *a = reinterpret_cast<cplx<R> *>(smem);
  cplx<R> *b = a + T * ld;
  const int kx0 = bx * T;
  const int nt = min(T, hx - kx0);
  cplx<R> *base = cm + (size_t)z * s2 * hx + kx0;
  Twiddle<R> *tw_s = reinterpret_cast<Twiddle<R> *>(b + T * ld);
  stage_twiddles(tw_s, tw, s2);
  // elements e = y T + c over the full tile width T; columns c >= nt (the
  // last tile) are skipped
  batched_copy(
      T * s2,
      [&](int e) {
        const int y = fdiv(e, V.f_fyT), c = e - y * T;
        return c < nt ? base[(size_t)y * hx + c] : cplx<R>{R(0), R(0)};
      },
      [&](int e, cplx<R> v) {
        const int y = fdiv(e, V.f_fyT), c = e - y * T;
        if (c < nt) a[c * ld + y] = v;
      });
  __syncthreads();
  cplx<R> *res = lds_fft(a, b, py, nt, ld, tw_s, inv != 0);
  for (int e = threadIdx.x; e < T * s2; e += blockDim.x) {
    const int y = fdiv(e, V.f_fyT), c = e - y * T;
    if (c < nt) base[(size_t)y * hx + c] = res[c * ld + y];
  }
}

// ----------------------------------------------- z pass with the convolution
// For every stored element (kx, ky, kz) the reference's CalcGIF loop counts
// |F|^2 * meshfac(nx,ny,nz) once, halved when kx is 0 or s1/2 (its
// energyfac halvings along y and z only undo double visits), with
// nx = kx, ny = min(ky, s2-ky), nz = min(kz, s3-kz); the virial uses
// (1 + 2 k^2 expf) on top (Src/energy.F90:6553-6578, 6994-7018).
// Tile of kx columns bx * fz_T, ... of line y: z forward, Green function,
// z inverse; the thread's energy and virial terms are added to esum, vsum.
template <typename R>
__device__ __forceinline__ void fftconv_tile(const SysDev &V, int bx, int y, int energy,
                                             char *smem, double &esum, double &vsum) {
  cplx<R> *__restrict__ cm = (cplx<R> *)V.mesh_c;
  const int s1 = V.sg.s[0], s2 = V.sg.s[1], s3 = V.sg.s[2], hx = V.hx, T = V.fz_T;
  const FftPlan &pz = V.plan[2];
  const Twiddle<R> *__restrict__ tw = (const Twiddle<R> *)V.tw[2];
  const SpmeAxes &ax = V.ax;
  const int ld = s3 + 1;
  cplx<R> *a = reinterpret_cast<cplx<R> *>(smem);
  cplx<R> *b = a + T * ld;
  const int kx0 = bx * T;
  const int nt = min(T, hx - kx0);
  const size_t zstride = (size_t)s2 * hx;
  cplx<R> *base = cm + (size_t)y * hx + kx0;
  Twiddle<R> *tw_s = reinterpret_cast<Twiddle<R> *>(b + T * ld);
  stage_twiddles(tw_s, tw, s3);
  batched_copy(
      T * s3,
      [&](int e) {
        const int z = fdiv(e, V.f_fzT), c = e - z * T;
        return c < nt ? base[z * zstride + c] : cplx<R>{R(0), R(0)};
      },
      [&](int e, cplx<R> v) {
        const int z = fdiv(e, V.f_fzT), c = e - z * T;
        if (c < nt) a[c * ld + z] = v;
      });
  __syncthreads();
  cplx<R> *f = lds_fft(a, b, pz, nt, ld, tw_s, false);
  const int ny = min(y, s2 - y);
  const double gy = ax.g[1][ny], kky = ax.kk[1][ny];
  for (int e = threadIdx.x; e < nt * s3; e += blockDim.x) {
    const int c = fdiv(e, V.f_s3), z = e - c * s3;
    const int nx = kx0 + c, nz = min(z, s3 - z);
    const double m2 = ax.kk[0][nx] + kky + ax.kk[2][nz];
    double mf = 0.0;
    if (m2 > 0.0) mf = ax.fac0 * ax.g[0][nx] * gy * ax.g[2][nz] / m2;
    cplx<R> v = f[c * ld + z];
    if (energy) {
      const double q2 = (double)v.x * (double)v.x + (double)v.y * (double)v.y;
      const double w = (nx == 0 || 2 * nx == s1) ? 0.5 : 1.0;
      esum += w * q2 * mf;
      vsum -= w * q2 * (1.0 + 2.0 * m2 * ax.expf) * mf;
    }
    const R mfr = (R)mf;
    f[c * ld + z] = {v.x * mfr, v.y * mfr};
  }
  __syncthreads();
  cplx<R> *g = (f == a) ? b : a;
  cplx<R> *res = lds_fft(f, g, pz, nt, ld, tw_s, true);
  for (int e = threadIdx.x; e < T * s3; e += blockDim.x) {
    const int z = fdiv(e, V.f_fzT), c = e - z * T;
    if (c < nt) base[z * zstride + c] = res[c * ld + z];
  }
}

// The z forward transform alone (no Green function), for the MC trial
// moves' kept spectrum: tile of kx columns bx * fz_T, ... of line y, read
// from the complex mesh and written, transformed, to out (same layout) as
// values of type O.
template <typename R, typename O>
__device__ __forceinline__ void fftz_fwd_tile(const SysDev &V, int bx, int y, cplx<O> *out,
                                              char *smem) {
  const cplx<R> *__restrict__ cm = (const cplx<R> *)V.mesh_c;
  const int s2 = V.sg.s[1], s3 = V.sg.s[2], hx = V.hx, T = V.fz_T;
  const FftPlan &pz = V.plan[2];
  const Twiddle<R> *__restrict__ tw = (const Twiddle<R> *)V.tw[2];
  const int ld = s3 + 1;
  cplx<R> *a = reinterpret_cast<cplx<R> *>(smem);
  cplx<R> *b = a + T * ld;
  const int kx0 = bx * T;
  const int nt = min(T, hx - kx0);
  const size_t zstride = (size_t)s2 * hx;
  const cplx<R> *base = cm + (size_t)y * hx + kx0;
  cplx<O> *obase = out + (size_t)y * hx + kx0;
  Twiddle<R> *tw_s = reinterpret_cast<Twiddle<R> *>(b + T * ld);
  stage_twiddles(tw_s, tw, s3);
  batched_copy(
      T * s3,
      [&](int e) {
        const int z = fdiv(e, V.f_fzT), c = e - z * T;
        return c < nt ? base[z * zstride + c] : cplx<R>{R(0), R(0)};
      },
      [&](int e, cplx<R> v) {
        const int z = fdiv(e, V.f_fzT), c = e - z * T;
        if (c < nt) a[c * ld + z] = v;
      });
  __syncthreads();
  const cplx<R> *f = lds_fft(a, b, pz, nt, ld, tw_s, false);
  for (int e = threadIdx.x; e < T * s3; e += blockDim.x) {
    const int z = fdiv(e, V.f_fzT), c = e - z * T;
    if (c < nt) {
      const cplx<R> v = f[c * ld + z];
      obase[z * zstride + c] = cplx<O>{(O)v.x, (O)v.y};
    }
  }
}

// ------------------------------------------- whole planes and lines (LDS)
// The same transforms over larger LDS tiles, for a workgroup that runs all
// passes of one replica: every kx column of planes z0 .. z0 + nz - 1 along
// y, of lines y0 .. y0 + ny - 1 along z.  In the complex mesh such a range
// is contiguous (planes) or nz runs of ny * hx elements (lines).
template <typename R>
__device__ __forceinline__ void ffty_planes(const SysDev &V, int z0, int nz, int inv,
                                            char *smem) {
  cplx<R> *__restrict__ base = (cplx<R> *)V.mesh_c + (size_t)z0 * V.sg.s[1] * V.hx;
  const int s2 = V.sg.s[1], hx = V.hx;
  const FftPlan &py = V.plan[1];
  const int ld = s2 + 1, nseq = nz * hx;
  cplx<R> *a = reinterpret_cast<cplx<R> *>(smem);
  cplx<R> *b = a + nseq * ld;
  Twiddle<R> *tw_s = reinterpret_cast<Twiddle<R> *>(b + nseq * ld);
  stage_twiddles(tw_s, (const Twiddle<R> *)V.tw[1], s2);
  // element e = (zz s2 + y) hx + kx of the range
  batched_copy(
      nseq * s2, [&](int e) { return base[e]; },
      [&](int e, cplx<R> v) {
        const int q = fdiv(e, V.f_hx), kx = e - q * hx;
        const int zz = fdiv(q, V.f_s2), y = q - zz * s2;
        a[(zz * hx + kx) * ld + y] = v;
      });
  __syncthreads();
  cplx<R> *res = lds_fft(a, b, py, nseq, ld, tw_s, inv != 0);
  for (int e = threadIdx.x; e < nseq * s2; e += blockDim.x) {
    const int q = fdiv(e, V.f_hx), kx = e - q * hx;
    const int zz = fdiv(q, V.f_s2), y = q - zz * s2;
    base[e] = res[(zz * hx + kx) * ld + y];
  }
}

template <typename R>
__device__ __forceinline__ void fftconv_lines(const SysDev &V, int y0, int ny, int energy,
                                              char *smem, double &esum, double &vsum) {
  cplx<R> *__restrict__ cm = (cplx<R> *)V.mesh_c;
  const int s1 = V.sg.s[0], s2 = V.sg.s[1], s3 = V.sg.s[2], hx = V.hx;
  const FftPlan &pz = V.plan[2];
  const SpmeAxes &ax = V.ax;
  const int ld = s3 + 1, nseq = ny * hx;
  cplx<R> *a = reinterpret_cast<cplx<R> *>(smem);
  cplx<R> *b = a + nseq * ld;
  Twiddle<R> *tw_s = reinterpret_cast<Twiddle<R> *>(b + nseq * ld);
  stage_twiddles(tw_s, (const Twiddle<R> *)V.tw[2], s3);
  const size_t zstride = (size_t)s2 * hx;
  cplx<R> *base = cm + (size_t)y0 * hx;
  // element e = z nseq + (yy hx + kx): sequence c = yy hx + kx, position z
  batched_copy(
      nseq * s3,
      [&](int e) {
        const int z = e / nseq, c = e - z * nseq;
        return base[z * zstride + c];
      },
      [&](int e, cplx<R> v) {
        const int z = e / nseq, c = e - z * nseq;
        a[c * ld + z] = v;
      });
  __syncthreads();
  cplx<R> *f = lds_fft(a, b, pz, nseq, ld, tw_s, false);
  for (int e = threadIdx.x; e < nseq * s3; e += blockDim.x) {
    const int c = fdiv(e, V.f_s3), z = e - c * s3;
    const int yy = fdiv(c, V.f_hx), nx = c - yy * hx;
    const int y = y0 + yy, nyy = min(y, s2 - y), nz = min(z, s3 - z);
    const double m2 = ax.kk[0][nx] + ax.kk[1][nyy] + ax.kk[2][nz];
    double mf = 0.0;
    if (m2 > 0.0) mf = ax.fac0 * ax.g[0][nx] * ax.g[1][nyy] * ax.g[2][nz] / m2;
    cplx<R> v = f[c * ld + z];
    if (energy) {
      const double q2 = (double)v.x * (double)v.x + (double)v.y * (double)v.y;
      const double w = (nx == 0 || 2 * nx == s1) ? 0.5 : 1.0;
      esum += w * q2 * mf;
      vsum -= w * q2 * (1.0 + 2.0 * m2 * ax.expf) * mf;
    }
    const R mfr = (R)mf;
    f[c * ld + z] = {v.x * mfr, v.y * mfr};
  }
  __syncthreads();
  cplx<R> *g = (f == a) ? b : a;
  cplx<R> *res = lds_fft(f, g, pz, nseq, ld, tw_s, true);
  for (int e = threadIdx.x; e < nseq * s3; e += blockDim.x) {
    const int z = e / nseq, c = e - z * nseq;
    base[z * zstride + c] = res[c * ld + z];
  }
}

}  // namespace
}  // namespace mfe
