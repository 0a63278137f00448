// Multi-dimensional complex FFT and DFT-domain circular convolution
// (scico/linop/_circconv.py:79-209) for gfx950.
//
// Layout: data (B, F0, ..., F{d-1}) row-major, B = product of the leading
// non-transformed axes, d <= 3 transformed axes.  One kernel performs one
// pass of 1D transforms along one axis; each workgroup loads LPB lines
// into LDS, transforms them by Stockham stages and writes them back:
//   * power-of-two lengths <= 4096: radix 16 after one stage of radix 2, 4
//     or 8;
//   * other lengths <= 512: mixed radix (Stages): powers of two up to 8, 3,
//     5 and 7 in registers, a larger prime factor p as p-term sums.
// Twiddles are float32 roundings of float64 exp(-2 pi i k / n).
// Inverse passes scale by 1/n, like numpy / jax ifft.
//
// Convolution y = real(ifftn(H * fftn(x))): forward passes on F{d-1} ..
// F1, one fused pass on F0 (forward, multiply by H or conj(H), inverse),
// inverse passes on F1 .. F{d-1}; the first pass reads the real input and
// the last one writes the real part.  With d == 1 the single fused pass
// does both.
//
// Real convolution over two axes (the deconvolution workload) runs on half
// spectra instead: rows transformed two real rows per complex
// FFT into (F1/2 + 1)-wide half spectra, one fused pass on those columns
// with the Hermitian part of H, rows inverted back to real.  At 1024 x 1024
// each line is one 256-thread workgroup's registers (four values per
// thread, radix-4 Stockham stages exchanged through LDS).
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <vector>

#include "apgm_stats.h"
#include "common.h"

using namespace scxr;

namespace scxr {
namespace fft {

constexpr int MAX_POW2 = 4096;
constexpr int MAX_DFT = 512;

// Stockham stages of a length that is no power of two, in order: stage s
// has radix R[s], with Ns = R[0] ... R[s - 1] before it.  mns / mnb are
// ceil(2^32 / Ns) and ceil(2^32 / (n / R)): the quotients of the stage's
// indices (below 2^13, by divisors below 2^10) are exact high words.
constexpr int MAX_STAGES = 8;
struct Stages {
  int count = 0;
  int twlds = 0;  // 1: a stage takes p-term sums, whose twiddles go to LDS
  int R[MAX_STAGES] = {};
  uint32_t mns[MAX_STAGES] = {};
  uint32_t mnb[MAX_STAGES] = {};
};

struct Pass {
  int n, log2n;          // line length, log2 (pow2) or -1 (mixed radix)
  long long stride;      // element stride along the line
  long long inner;       // lines per outer index (= stride)
  long long lines;       // total lines
  int lpb;               // lines per workgroup
  int in_real;           // input is real float32
  int out_real;          // output real part (float32)
  int inverse;           // direction of the (non-fused) transform
  int fused;             // forward, multiply by h (conj if conj_h), inverse
  int conj_h;
  const float2* tw;      // n twiddles exp(-2 pi i k / n)
  const float2* h;       // fused: spectrum, indexed by k * stride + inner
};

__device__ __forceinline__ float2 cmul(float2 a, float2 b) {
  return make_float2(__fsub_rn(__fmul_rn(a.x, b.x), __fmul_rn(a.y, b.y)),
                     __fadd_rn(__fmul_rn(a.x, b.y), __fmul_rn(a.y, b.x)));
}

__device__ __forceinline__ float2 conjf2(float2 a) { return make_float2(a.x, -a.y); }

// The same in float64, for the spectra that a solver prepares once.
__device__ __forceinline__ double2 cmul(double2 a, double2 b) {
  return make_double2(a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x);
}
__device__ __forceinline__ double2 conjf2(double2 a) { return make_double2(a.x, -a.y); }
template <class V>
using Real = decltype(V::x);
template <class V>
__device__ __forceinline__ V cmake(Real<V> x, Real<V> y) {
  V v;
  v.x = x;
  v.y = y;
  return v;
}
__device__ __forceinline__ float fma_(float a, float b, float c) { return fmaf(a, b, c); }
__device__ __forceinline__ double fma_(double a, double b, double c) { return fma(a, b, c); }

// Power-of-two lengths: Stockham auto-sort passes of radix 16 (after one
// pass of radix 2, 4 or 8 for log2 n mod 4) on lpb lines held in one LDS
// buffer.  Each
// thread takes whole butterflies: it reads its R inputs x[j + r n / R] into
// registers, twiddles them by w^(k r) (k = j mod Ns, w = exp(-2 pi i /
// (R Ns)), taken from the n-entry table), transforms them and, after a
// barrier, writes them to x[(j / Ns) R Ns + k + r Ns]; the output is in
// natural order, so the fused convolution pass multiplies by the spectrum
// and runs the inverse stages on the same buffer.
constexpr int SH_THREADS = 256;
// Values per thread and stage: 4 for workgroups of at most 1024 values, else 32
// (lpb n <= 8192; powers of two).  The kernels unroll over them for every
// radix, and at 32 the mixed-radix column pass was 160 KB of code, which does
// not stay in the instruction cache (convolution of 3 x 360 x 480: 39 -> 25 us,
// 512 x 512: 27 -> 22 us).
constexpr int SH_MAXV = 32, SH_FEW = 4;

__device__ __forceinline__ float2 cadd(float2 a, float2 b) {
  return make_float2(__fadd_rn(a.x, b.x), __fadd_rn(a.y, b.y));
}
__device__ __forceinline__ float2 csub(float2 a, float2 b) {
  return make_float2(__fsub_rn(a.x, b.x), __fsub_rn(a.y, b.y));
}

__device__ __forceinline__ double2 cadd(double2 a, double2 b) {
  return make_double2(a.x + b.x, a.y + b.y);
}
__device__ __forceinline__ double2 csub(double2 a, double2 b) {
  return make_double2(a.x - b.x, a.y - b.y);
}

// 4-point DFT of a[0], a[s], a[2 s], a[3 s] in place (natural order).
template <int S, int N, class V>
__device__ __forceinline__ void dft4_strided(V (&v)[N], int o, bool inv) {
  const V s02 = cadd(v[o], v[o + 2 * S]), d02 = csub(v[o], v[o + 2 * S]);
  const V s13 = cadd(v[o + S], v[o + 3 * S]), d13 = csub(v[o + S], v[o + 3 * S]);
  // -i d13 (forward) or +i d13 (inverse)
  const V t = inv ? cmake<V>(-d13.y, d13.x) : cmake<V>(d13.y, -d13.x);
  v[o] = cadd(s02, s13);
  v[o + 2 * S] = csub(s02, s13);
  v[o + S] = cadd(d02, t);
  v[o + 3 * S] = csub(d02, t);
}

// exp(-2 pi i m / 16) = (cos(pi m / 8), -sin(pi m / 8)) for m = 0 .. 15,
// conjugated for the inverse: the internal twiddles of the 8- and 16-point
// butterflies (m is a compile-time constant there, so the tables fold).
template <class V>
__device__ __forceinline__ V w16(int m, bool inv) {
  using T = Real<V>;
  constexpr T c1 = static_cast<T>(0.92387953251128674), s1 = static_cast<T>(0.38268343236508978);
  constexpr T h = static_cast<T>(0.70710678118654752), o = 1, z = 0;
  constexpr T cs[16] = {o, c1, h, s1, z, -s1, -h, -c1, -o, -c1, -h, -s1, z, s1, h, c1};
  constexpr T sn[16] = {z, s1, h, c1, o, c1, h, s1, z, -s1, -h, -c1, -o, -c1, -h, -s1};
  return cmake<V>(cs[m & 15], inv ? sn[m & 15] : -sn[m & 15]);
}

// cos and sin of 2 pi k / R for k <= R / 2: the odd butterflies' constants
// (indices are compile-time constants, so the tables fold).
template <int R>
struct OddTrig;
template <>
struct OddTrig<3> {
  static constexpr double cs[2] = {1.0, -0.5};
  static constexpr double sn[2] = {0.0, 0.86602540378443865};
};
template <>
struct OddTrig<5> {
  static constexpr double cs[3] = {1.0, 0.30901699437494742, -0.80901699437494742};
  static constexpr double sn[3] = {0.0, 0.95105651629515357, 0.58778525229247313};
};
template <>
struct OddTrig<7> {
  static constexpr double cs[4] = {1.0, 0.62348980185873353, -0.22252093395631440,
                                   -0.90096886790241913};
  static constexpr double sn[4] = {0.0, 0.78183148246802981, 0.97492791218182361,
                                   0.43388373911755812};
};

template <int R, class V>
__device__ __forceinline__ void dft_small(V (&v)[R], bool inv) {
  if constexpr (R == 16 || R == 8) {
    // R = 4 Q: inputs n1 + 4 n2 ... as R = Q x 4 with Q = R / 4:
    // DFT over the Q-strided groups, twiddle, then 4- (or 2-) point DFTs.
    constexpr int Q = R / 4;  // 4 (R = 16) or 2 (R = 8)
    // step 1: for each n1 < Q, 4-point DFT over n2 of v[n1 + Q n2]
#pragma unroll
    for (int n1 = 0; n1 < Q; ++n1) dft4_strided<Q, R>(v, n1, inv);
    // step 2: twiddle v[n1 + Q k2] by W_R^(n1 k2)
#pragma unroll
    for (int n1 = 1; n1 < Q; ++n1)
#pragma unroll
      for (int k2 = 1; k2 < 4; ++k2) v[n1 + Q * k2] = cmul(v[n1 + Q * k2], w16<V>(n1 * k2 * (16 / R), inv));
    // step 3: for each k2, Q-point DFT over n1; output k = k2 + 4 k1
    V o[R];
#pragma unroll
    for (int k2 = 0; k2 < 4; ++k2) {
      if constexpr (Q == 4) {
        V g[4] = {v[Q * k2], v[1 + Q * k2], v[2 + Q * k2], v[3 + Q * k2]};
        dft4_strided<1, 4>(g, 0, inv);
#pragma unroll
        for (int k1 = 0; k1 < 4; ++k1) o[k2 + 4 * k1] = g[k1];
      } else {
        const V a = v[Q * k2], b = v[1 + Q * k2];
        o[k2] = cadd(a, b);
        o[k2 + 4] = csub(a, b);
      }
    }
#pragma unroll
    for (int r = 0; r < R; ++r) v[r] = o[r];
  } else if constexpr (R == 3 || R == 5 || R == 7) {
    // odd R: with s_k = x_k + x_{R-k}, d_k = x_k - x_{R-k},
    // X_m, X_{R-m} = x_0 + sum_k cos(2 pi k m / R) s_k
    //                -+ i sum_k sin(2 pi k m / R) d_k
    constexpr int H = R / 2;
    V sm[H], df[H];
    V x0 = v[0];
#pragma unroll
    for (int k = 1; k <= H; ++k) {
      sm[k - 1] = cadd(v[k], v[R - k]);
      df[k - 1] = csub(v[k], v[R - k]);
      x0 = cadd(x0, sm[k - 1]);
    }
    V o[R];
    o[0] = x0;
#pragma unroll
    for (int m = 1; m <= H; ++m) {
      V c = v[0], d = cmake<V>(0, 0);
#pragma unroll
      for (int k = 1; k <= H; ++k) {
        const int t = (k * m) % R;  // a compile-time constant once unrolled
        using T = Real<V>;
        const T co = static_cast<T>(OddTrig<R>::cs[t <= H ? t : R - t]);
        const T si = static_cast<T>(t <= H ? OddTrig<R>::sn[t] : -OddTrig<R>::sn[R - t]);
        c = cmake<V>(fma_(co, sm[k - 1].x, c.x), fma_(co, sm[k - 1].y, c.y));
        d = cmake<V>(fma_(si, df[k - 1].x, d.x), fma_(si, df[k - 1].y, d.y));
      }
      // -i d (forward) or +i d (inverse)
      const V t = inv ? cmake<V>(-d.y, d.x) : cmake<V>(d.y, -d.x);
      o[m] = cadd(c, t);
      o[R - m] = csub(c, t);
    }
#pragma unroll
    for (int r = 0; r < R; ++r) v[r] = o[r];
  } else if constexpr (R == 2) {
    const V a = v[0], b = v[1];
    v[0] = cadd(a, b);
    v[1] = csub(a, b);
  } else {
    dft4_strided<1, 4>(v, 0, inv);
  }
}

template <int R, int MAXV>
__device__ __forceinline__ void stockham_stage(float2* X, int n, int lpb, int Ns,
                                               const float2* tw, bool inv) {
  const int nb = n / R, tot = lpb * nb;  // butterflies
  const int tstep = n / (R * Ns);
  constexpr int NQ = (MAXV + R - 1) / R;
  float2 v[NQ][R];
  int dst[NQ];
#pragma unroll
  for (int q = 0; q < NQ; ++q) {
    const int b = threadIdx.x + q * SH_THREADS;
    dst[q] = -1;
    if (b < tot) {
      const int l = b / nb, j = b - l * nb;
      float2* x = X + l * n;
      const int k = j & (Ns - 1);
#pragma unroll
      for (int r = 0; r < R; ++r) v[q][r] = x[j + r * nb];
#pragma unroll
      for (int r = 1; r < R; ++r) {
        float2 w = tw[(k * r * tstep) & (n - 1)];
        if (inv) w = conjf2(w);
        v[q][r] = cmul(v[q][r], w);
      }
      dft_small<R>(v[q], inv);
      dst[q] = l * n + (j - k) * R + k;
    }
  }
  __syncthreads();
#pragma unroll
  for (int q = 0; q < NQ; ++q) {
    if (dst[q] >= 0) {
#pragma unroll
      for (int r = 0; r < R; ++r) X[dst[q] + r * Ns] = v[q][r];
    }
  }
  __syncthreads();
}

template <int MAXV>
__device__ __forceinline__ void stockham(float2* X, int n, int log2n, int lpb,
                                         const float2* tw, bool inv) {
  // one stage of radix 2, 4 or 8 for log2 n mod 4, then radix-16 stages
  int Ns = 1;
  switch (log2n & 3) {
    case 1: stockham_stage<2, MAXV>(X, n, lpb, Ns, tw, inv); Ns = 2; break;
    case 2: stockham_stage<4, MAXV>(X, n, lpb, Ns, tw, inv); Ns = 4; break;
    case 3: stockham_stage<8, MAXV>(X, n, lpb, Ns, tw, inv); Ns = 8; break;
    default: break;
  }
  for (; Ns < n; Ns *= 16) stockham_stage<16, MAXV>(X, n, lpb, Ns, tw, inv);
}

// Mixed radix for lengths that are no power of two.  Bound by the latency
// of the stages' LDS round trips and barriers (n log n work is small): 540
// row pairs of 480 points 7.5 us, 723 half-spectrum columns of 360 (forward,
// spectrum, inverse) 12.8 us.  Sums over all n inputs, which these lengths
// took before, cost 454 us a pass on the full spectrum: 3 x 360 x 480
// convolution 1380 -> 25 us, and its error against float64 1.7e-6 -> 1.7e-7.
//
// One stage: as stockham_stage, with the quotients by Ns and n / R taken as high words of the stage's magic
// factors (k r tstep < n, so the twiddle index needs no reduction).
template <int R, int MAXV, class V>
__device__ __forceinline__ void mixed_stage(V* X, int n, int lpb, int Ns, uint32_t mns,
                                            uint32_t mnb, const V* tw, bool inv) {
  constexpr int NQ = (MAXV + R - 1) / R;
  const int nb = n / R, tot = lpb * nb;  // butterflies
  const int tstep = n / (R * Ns);
  V v[NQ][R];
  int dst[NQ];
#pragma unroll
  for (int q = 0; q < NQ; ++q) {
    const int b = threadIdx.x + q * SH_THREADS;
    dst[q] = -1;
    if (b < tot) {
      const int l = nb > 1 ? static_cast<int>(__umulhi(b, mnb)) : b, j = b - l * nb;
      const int g = Ns > 1 ? static_cast<int>(__umulhi(j, mns)) : j, k = j - g * Ns;
      const V* x = X + l * n + j;
#pragma unroll
      for (int r = 0; r < R; ++r) v[q][r] = x[r * nb];
      if (Ns > 1) {
#pragma unroll
        for (int r = 1; r < R; ++r) {
          V w = tw[k * r * tstep];
          if (inv) w = conjf2(w);
          v[q][r] = cmul(v[q][r], w);
        }
      }
      dft_small<R>(v[q], inv);
      dst[q] = l * n + g * R * Ns + k;
    }
  }
  __syncthreads();
#pragma unroll
  for (int q = 0; q < NQ; ++q) {
    if (dst[q] >= 0) {
#pragma unroll
      for (int r = 0; r < R; ++r) X[dst[q] + r * Ns] = v[q][r];
    }
  }
  __syncthreads();
}

// A stage of any radix R (a prime above 7): output s of butterfly j is the
// R-term sum of x[j + r n / R] w^(r (k tstep + s n / R)), w = exp(-2 pi i /
// n), from the n twiddles in LDS.
template <int MAXV, class V>
__device__ __forceinline__ void prime_stage(V* X, int n, int lpb, int R, int Ns, uint32_t mns,
                                            uint32_t mnb, const V* tw, bool inv) {
  const int nb = n / R, tot = lpb * n;
  const int tstep = n / (R * Ns);
  V o[MAXV];
  // element e = (line l, output s, butterfly j), j fastest
  auto where = [&](int e, int& l, int& s, int& g, int& k) {
    const int ls = nb > 1 ? static_cast<int>(__umulhi(e, mnb)) : e, j = e - ls * nb;
    l = ls / R;
    s = ls - l * R;
    g = Ns > 1 ? static_cast<int>(__umulhi(j, mns)) : j;
    k = j - g * Ns;
  };
#pragma unroll
  for (int q = 0; q < MAXV; ++q) {
    const int e = threadIdx.x + q * SH_THREADS;
    if (e < tot) {
      int l, s, g, k;
      where(e, l, s, g, k);
      const V* x = X + l * n + g * Ns + k;
      int step = k * tstep + s * nb, idx = step;
      if (step >= n) idx = step -= n;
      // Term 0 has weight 1.  The R - 1 others (an even number) are added in two
      // halves, and each half's four kinds of product apart, with one rounding
      // per product and sum.  One chain of rounded products left the convolution
      // on half spectra, whose rows come in pairs, further off than sums over
      // the full spectrum: 509 x 503 8.2e-7 against 7.4e-7 of the result, 5.8e-7
      // with these.
      Real<V> xx[2] = {x[0].x, 0}, yy[2] = {0, 0}, xy[2] = {0, 0}, yx[2] = {x[0].y, 0};
      for (int r = 1; r < R; r += 2) {
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          V w = tw[idx];
          if (inv) w = conjf2(w);
          const V a = x[(r + h) * nb];
          xx[h] = fma_(a.x, w.x, xx[h]);
          yy[h] = fma_(a.y, w.y, yy[h]);
          xy[h] = fma_(a.x, w.y, xy[h]);
          yx[h] = fma_(a.y, w.x, yx[h]);
          idx += step;
          if (idx >= n) idx -= n;
        }
      }
      o[q] = cmake<V>((xx[0] + xx[1]) - (yy[0] + yy[1]), (xy[0] + xy[1]) + (yx[0] + yx[1]));
    }
  }
  __syncthreads();
#pragma unroll
  for (int q = 0; q < MAXV; ++q) {
    const int e = threadIdx.x + q * SH_THREADS;
    if (e < tot) {
      int l, s, g, k;
      where(e, l, s, g, k);
      X[l * n + g * R * Ns + k + s * Ns] = o[q];
    }
  }
  __syncthreads();
}

// Mixed-radix transform of lpb lines in X; tw in LDS if S.twlds.
template <int MAXV, class V>
__device__ __forceinline__ void mixed(V* X, int n, const Stages& S, int lpb, const V* tw,
                                      bool inv) {
  int Ns = 1;
  for (int s = 0; s < S.count; ++s) {
    const int R = S.R[s];
    const uint32_t mns = S.mns[s], mnb = S.mnb[s];
    switch (R) {
      case 2: mixed_stage<2, MAXV>(X, n, lpb, Ns, mns, mnb, tw, inv); break;
      case 3: mixed_stage<3, MAXV>(X, n, lpb, Ns, mns, mnb, tw, inv); break;
      case 4: mixed_stage<4, MAXV>(X, n, lpb, Ns, mns, mnb, tw, inv); break;
      case 5: mixed_stage<5, MAXV>(X, n, lpb, Ns, mns, mnb, tw, inv); break;
      case 7: mixed_stage<7, MAXV>(X, n, lpb, Ns, mns, mnb, tw, inv); break;
      case 8: mixed_stage<8, MAXV>(X, n, lpb, Ns, mns, mnb, tw, inv); break;
      default: prime_stage<MAXV>(X, n, lpb, R, Ns, mns, mnb, tw, inv);
    }
    Ns *= R;
  }
}

// The transform of a pass's lines, by length.
template <bool MIXED, int MAXV>
__device__ __forceinline__ void transform(float2* X, int n, int log2n, const Stages& S, int lpb,
                                          const float2* tw, bool inv) {
  if constexpr (MIXED)
    mixed<MAXV>(X, n, S, lpb, tw, inv);
  else
    stockham<MAXV>(X, n, log2n, lpb, tw, inv);
}

// Twiddles of a mixed pass: copied behind the tot LDS values when a stage
// reads one per term, else read from the table (it stays in the vector
// cache).
template <bool MIXED>
__device__ __forceinline__ const float2* pass_twiddles(float2* X, int tot, int n,
                                                       const Stages& S, const float2* tw) {
  if (!MIXED || !S.twlds) return tw;
  for (int k = threadIdx.x; k < n; k += SH_THREADS) X[tot + k] = tw[k];
  return X + tot;
}

// At least four waves per SIMD: with 131 registers, above the 128 that allow
// them, 1000 and 4000 lines of 2048 took 34.5 and 107 us against 26.5 and 92.
template <bool MIXED, int MAXV>
__global__ __launch_bounds__(SH_THREADS) __attribute__((amdgpu_waves_per_eu(4))) void
stockham_kernel(const void* __restrict__ in,
                                                              void* __restrict__ out, Pass P,
                                                              Stages S, float scale,
                                                              const int32_t* pred) {
  if (pred_off(pred)) return;
  extern __shared__ float2 lds[];  // lpb * n values (and n twiddles, S.twlds)
  __shared__ long long base[64];
  __shared__ long long hoff[64];  // spectrum offset of each line (fused pass)
  const int n = P.n, lpb = P.lpb, tot = lpb * n;
  float2* X = lds;
  // twiddles are read from the n-entry table in global memory (it stays in
  // the vector cache; staging it in LDS per workgroup cost more)
  const float2* twl = pass_twiddles<MIXED>(X, tot, n, S, P.tw);
  const bool contiguous = P.stride == 1;
  // Strided passes: workgroups dispatched to one XCD (consecutive ids go to
  // the 8 XCDs in turn) take consecutive line groups, so the cache lines
  // that neighbouring columns share stay in that XCD's L2.
  long long blk = blockIdx.x;
  // (a bijection of the first 8 * floor(G / 8) workgroups; the rest keep
  // their own line group)
  if (!contiguous) {
    const long long G8 = (static_cast<long long>(gridDim.x) / 8) * 8;
    if (blk < G8) blk = (blk % 8) * (G8 / 8) + blk / 8;
  }
  const long long line0 = blk * lpb;
  const int nl = static_cast<int>(min(static_cast<long long>(lpb), P.lines - line0));
  if (threadIdx.x < lpb) {
    const long long L = line0 + threadIdx.x;
    const long long outer = L / P.inner, inr = L - outer * P.inner;
    base[threadIdx.x] = outer * n * P.stride + inr;
    hoff[threadIdx.x] = inr;
  }
  __syncthreads();
  auto split = [&](int e, int& l, int& k) {
    if (contiguous) {
      l = e / n;
      k = e - l * n;
    } else {
      k = e / lpb;
      l = e - k * lpb;
    }
  };
  {
    // every load of the thread is issued before the first LDS store
    float2 vv[MAXV];
#pragma unroll
    for (int q = 0; q < MAXV; ++q) {
      const int e = threadIdx.x + q * SH_THREADS;
      if (e < tot) {
        int l, k;
        split(e, l, k);
        float2 v = make_float2(0.0f, 0.0f);
        if (l < nl) {
          const long long g = base[l] + static_cast<long long>(k) * P.stride;
          v = P.in_real ? make_float2(static_cast<const float*>(in)[g], 0.0f)
                        : static_cast<const float2*>(in)[g];
        }
        vv[q] = v;
      }
    }
#pragma unroll
    for (int q = 0; q < MAXV; ++q) {
      const int e = threadIdx.x + q * SH_THREADS;
      if (e < tot) {
        int l, k;
        split(e, l, k);
        X[l * n + k] = vv[q];
      }
    }
  }
  constexpr bool AHEAD = MAXV <= SH_FEW;  // the spectrum is loaded before the transform
  float2 hv[AHEAD ? MAXV : 1];
  auto spectrum = [&](int e) {
    const int l = e / n, k = e - l * n;
    return l < nl ? P.h[static_cast<long long>(k) * P.stride + hoff[l]] : make_float2(0.0f, 0.0f);
  };
  if constexpr (AHEAD) {
    if (P.fused) {
#pragma unroll
      for (int q = 0; q < MAXV; ++q)
        if (threadIdx.x + q * SH_THREADS < tot) hv[q] = spectrum(threadIdx.x + q * SH_THREADS);
    }
  }
  __syncthreads();
  transform<MIXED, MAXV>(X, n, P.log2n, S, lpb, twl, P.fused ? false : (P.inverse != 0));
  if (P.fused) {
    auto times = [&](int e, float2 h) {
      if (P.conj_h) h = conjf2(h);
      X[e] = cmul(h, X[e]);
    };
    if constexpr (AHEAD) {
#pragma unroll
      for (int q = 0; q < MAXV; ++q)
        if (threadIdx.x + q * SH_THREADS < tot)
          times(threadIdx.x + q * SH_THREADS, hv[q]);
    } else {
      for (int e = threadIdx.x; e < tot; e += SH_THREADS)
        if (e / n < nl) times(e, spectrum(e));
    }
    __syncthreads();
    transform<MIXED, MAXV>(X, n, P.log2n, S, lpb, twl, true);
  }
  for (int e = threadIdx.x; e < tot; e += SH_THREADS) {
    int l, k;
    split(e, l, k);
    if (l < nl) {
      const long long g = base[l] + static_cast<long long>(k) * P.stride;
      const float2 v = X[l * n + k];
      if (P.out_real)
        static_cast<float*>(out)[g] = __fmul_rn(v.x, scale);
      else
        static_cast<float2*>(out)[g] = make_float2(__fmul_rn(v.x, scale), __fmul_rn(v.y, scale));
    }
  }
}

// ------------------------------------------- real 2D convolution path --
//
// For two FFT axes (F0, F1) the convolution of real data runs on half
// spectra.  Rows are transformed two at a time: z = x_a + i x_b
// has the DFT Z = X_a + i X_b with X_a, X_b Hermitian, so
//   X_a[k] = (Z[k] + conj(Z[-k])) / 2,   X_b[k] = (Z[k] - conj(Z[-k])) / (2 i),
// and only k = 0 .. F1/2 of each row is kept (H1 = F1/2 + 1 columns).  The
// columns of that half spectrum take the fused pass (forward, times the
// spectrum, inverse).  real(ifft2(H X)) = irfft2(Hs X) with the Hermitian
// part Hs[k] = (H[k] + conj(H[-k])) / 2 of H (equal to H for a real
// kernel), so the plan keeps Hs on the half grid.  The inverse rows rebuild
// Z = X_a + i X_b on the full row from the Hermitian extensions (the
// imaginary parts of the k = 0 and, for even F1, k = F1/2 bins dropped, as
// irfft does) and write x_a = Re z, x_b = Im z.

// The row pairs of a pass over R rows.  A pair shares its rounding (and
// whatever is not finite), so both rows come from one image: where the images
// of a batch have an odd number of rows, `odd` is the number of pairs of an
// image, the last of which is one row alone (0: rows pair throughout).  ODD
// is a template parameter of the kernels: a branch per value kept their loads
// from being in flight together (64 x 2048: 25.7 -> 31.3 us).
struct RowPairs {
  long long R;
  unsigned odd;
};
// First row of a pair, and its second (R or more: there is none).
template <bool ODD>
__device__ __forceinline__ void pair_rows(const RowPairs& P, long long pair, long long& ra,
                                          long long& rb) {
  ra = 2 * pair;
  rb = ra + 1;
  if constexpr (ODD) {
    const unsigned q = static_cast<unsigned>(pair), im = q / P.odd;
    ra -= im;
    rb = q - im * P.odd == P.odd - 1 ? P.R : ra + 1;
  }
}

// Forward rows: real x (R rows of n) -> half spectra (R rows of n/2 + 1).
template <bool MIXED, int MAXV, bool ODD>
__global__ __launch_bounds__(SH_THREADS) void r2c_rows_kernel(const float* __restrict__ x,
                                                              float2* __restrict__ half, int n,
                                                              int log2n, Stages S, RowPairs P,
                                                              int lpb,
                                                              const float2* __restrict__ tw,
                                                              const int32_t* pred) {
  if (pred_off(pred)) return;
  extern __shared__ float2 lds[];  // lpb * n values
  float2* X = lds;
  const int tot = lpb * n, H1 = n / 2 + 1;
  const float2* twl = pass_twiddles<MIXED>(X, tot, n, S, tw);
  const long long R = P.R, pair0 = static_cast<long long>(blockIdx.x) * lpb;
  {
    float2 vv[MAXV];
#pragma unroll
    for (int q = 0; q < MAXV; ++q) {
      const int e = threadIdx.x + q * SH_THREADS;
      if (e < tot) {
        const int l = e / n, k = e - l * n;
        long long ra, rb;
        pair_rows<ODD>(P, pair0 + l, ra, rb);
        const float a = ra < R ? x[ra * n + k] : 0.0f;
        const float b = rb < R ? x[rb * n + k] : 0.0f;
        vv[q] = make_float2(a, b);
      }
    }
#pragma unroll
    for (int q = 0; q < MAXV; ++q) {
      const int e = threadIdx.x + q * SH_THREADS;
      if (e < tot) X[e] = vv[q];
    }
  }
  __syncthreads();
  transform<MIXED, MAXV>(X, n, log2n, S, lpb, twl, false);
  for (int e = threadIdx.x; e < lpb * H1; e += SH_THREADS) {
    const int l = e / H1, k = e - l * H1;
    long long ra, rb;
    pair_rows<ODD>(P, pair0 + l, ra, rb);
    const float2 zk = X[l * n + k], zm = X[l * n + (k ? n - k : 0)];
    if (ra < R)
      half[ra * H1 + k] = make_float2(__fmul_rn(0.5f, __fadd_rn(zk.x, zm.x)),
                                      __fmul_rn(0.5f, __fsub_rn(zk.y, zm.y)));
    if (rb < R)
      half[rb * H1 + k] = make_float2(__fmul_rn(0.5f, __fadd_rn(zk.y, zm.y)),
                                      __fmul_rn(0.5f, __fsub_rn(zm.x, zk.x)));
  }
}

// Inverse rows: half spectra (R rows of n/2 + 1) of the row pairs pair0 + l ->
// transformed lines X (the real rows of each pair, unscaled).
template <bool MIXED, int MAXV, bool ODD>
__device__ __forceinline__ void c2r_lines(const float2* __restrict__ half, float2* X, int n,
                                          int log2n, const Stages& S, const RowPairs& P, int lpb,
                                          long long pair0, const float2* __restrict__ tw) {
  const int H1 = n / 2 + 1;
  const long long R = P.R;
  const float2* twl = pass_twiddles<MIXED>(X, lpb * n, n, S, tw);
  for (int e = threadIdx.x; e < lpb * H1; e += SH_THREADS) {
    const int l = e / H1, k = e - l * H1;
    long long ra, rb;
    pair_rows<ODD>(P, pair0 + l, ra, rb);
    float2 a = ra < R ? half[ra * H1 + k] : make_float2(0.0f, 0.0f);
    float2 b = rb < R ? half[rb * H1 + k] : make_float2(0.0f, 0.0f);
    if (k == 0 || 2 * k == n) a.y = b.y = 0.0f;
    // Z[k] = A[k] + i B[k];  Z[n - k] = conj(A[k]) + i conj(B[k])
    X[l * n + k] = make_float2(__fsub_rn(a.x, b.y), __fadd_rn(a.y, b.x));
    if (k > 0 && 2 * k < n) X[l * n + n - k] = make_float2(__fadd_rn(a.x, b.y), __fsub_rn(b.x, a.y));
  }
  __syncthreads();
  transform<MIXED, MAXV>(X, n, log2n, S, lpb, twl, true);
}

// Inverse rows to real y (R rows of n), times scale.
template <bool MIXED, int MAXV, bool ODD>
__global__ __launch_bounds__(SH_THREADS) void c2r_rows_kernel(const float2* __restrict__ half,
                                                              float* __restrict__ y, int n,
                                                              int log2n, Stages S, RowPairs P,
                                                              int lpb,
                                                              const float2* __restrict__ tw,
                                                              float scale, const int32_t* pred) {
  if (pred_off(pred)) return;
  extern __shared__ float2 lds[];
  float2* X = lds;
  const long long R = P.R, pair0 = static_cast<long long>(blockIdx.x) * lpb;
  c2r_lines<MIXED, MAXV, ODD>(half, X, n, log2n, S, P, lpb, pair0, tw);
  for (int e = threadIdx.x; e < lpb * n; e += SH_THREADS) {
    const int l = e / n, k = e - l * n;
    long long ra, rb;
    pair_rows<ODD>(P, pair0 + l, ra, rb);
    const float2 v = X[e];
    if (ra < R) y[ra * n + k] = __fmul_rn(v.x, scale);
    if (rb < R) y[rb * n + k] = __fmul_rn(v.y, scale);
  }
}

// ------------------------------- 1024-point lines on 256 threads --------
//
// Radix-4 Stockham transform of one 1024-point line by a 256-thread
// workgroup, four values per thread: thread j holds x[j + 256 r], r < 4,
// on entry and X[j + 256 r] on exit (natural order, no reordering pass).
// Stage s (Ns = 4^s, s < 5): twiddle a[r] by W_{4 Ns}^{r k}, k = j mod Ns
// (W = exp(-2 pi i / ...)), 4-point DFT over r, write a[r] to
// (j / Ns) 4 Ns + k + r Ns; the next stage reads positions j + 256 r.
// Stage 0 takes the registers as loaded and stage 4's outputs stay in
// registers, so a transform makes four LDS exchanges.  Four waves per line
// (2052 waves for the 513 columns of a 1024 x 1024 half spectrum) hide the
// latency that one wave per line leaves exposed.
constexpr int Q1K = 1024, QT = 256;
constexpr int Q_LDS = Q1K + Q1K / 16;  // padded line (float2)
__device__ __forceinline__ int q_pad(int i) { return i + (i >> 4); }

struct QTw {
  float2 w[4][3];  // stages 1..4, r = 1..3
};

__device__ __forceinline__ void q_twiddles(QTw& t, const float2* __restrict__ tw, int j) {
#pragma unroll
  for (int s = 1; s < 5; ++s) {
    const int Ns = 1 << (2 * s);
    const int k = j & (Ns - 1);
#pragma unroll
    for (int r = 1; r < 4; ++r) t.w[s - 1][r - 1] = tw[(r * k * (QT / Ns)) & (Q1K - 1)];
  }
}

// Transform of thread j's four values on the line buffer lds (every thread
// of the workgroup calls it: the barriers are workgroup wide).
template <bool INV>
__device__ __forceinline__ void q_fft(float2 (&a)[4], float2* lds, const QTw& t, int j) {
#pragma unroll
  for (int s = 0; s < 5; ++s) {
    const int Ns = 1 << (2 * s);
    if (s > 0) {
      __syncthreads();  // the previous stage's writes are visible
#pragma unroll
      for (int r = 0; r < 4; ++r) a[r] = lds[q_pad(j + QT * r)];
#pragma unroll
      for (int r = 1; r < 4; ++r)
        a[r] = cmul(a[r], INV ? conjf2(t.w[s - 1][r - 1]) : t.w[s - 1][r - 1]);
    }
    dft_small<4>(a, INV);
    if (s < 4) {
      const int base = (j >> (2 * s)) * 4 * Ns + (j & (Ns - 1));
      __syncthreads();  // every read of the buffer is done before it is overwritten
#pragma unroll
      for (int r = 0; r < 4; ++r) lds[q_pad(base + r * Ns)] = a[r];
    }
  }
}

// The 1024 x 1024 half spectrum is kept transposed, column k1 of every item
// contiguous: halfT[(item H1 + k1) 1024 + row], so that the column
// transforms read and write whole lines.  The row kernels take QR = 4 rows
// (two complex transforms, 512 threads) per workgroup and move each
// column's four values of those rows as two 16-byte pairs.
constexpr int QR = 4;
constexpr int QH1 = Q1K / 2 + 1;

// Row block of a row-kernel workgroup whose grid holds `first` other
// workgroups before its G row blocks: consecutive workgroups go to the 8
// XCDs in turn, so each XCD takes a run of neighbouring row blocks, whose
// pieces of one transposed column share cache lines (a bijection of the
// first 8 * floor(G / 8) row workgroups; the rest keep their own block).
__device__ __forceinline__ long long q_row_block(int first = 0) {
  long long b = static_cast<long long>(blockIdx.x) - first;
  const long long G8 = ((static_cast<long long>(gridDim.x) - first) / 8) * 8;
  if (b < G8) b = (b % 8) * (G8 / 8) + b / 8;
  return b;
}

// Forward rows: two real rows per complex transform (z = x_a + i x_b;
// X_a[k] = (Z[k] + conj Z[-k]) / 2, X_b[k] = (Z[k] - conj Z[-k]) / 2i).
__global__ __launch_bounds__(2 * QT) void q1k_r2c_kernel(const float* __restrict__ x,
                                                         float2* __restrict__ halfT,
                                                         const float2* __restrict__ tw,
                                                         const int32_t* pred) {
  if (pred_off(pred)) return;
  __shared__ float2 lds[2][Q_LDS];
  const int g = threadIdx.x >> 8, j = threadIdx.x & (QT - 1);
  const long long r0 = q_row_block() * QR;  // first row (all in one item)
  const long long ra = r0 + 2 * g;
  QTw t;
  q_twiddles(t, tw, j);
  float2 a[4];
#pragma unroll
  for (int r = 0; r < 4; ++r)
    a[r] = make_float2(x[ra * Q1K + j + QT * r], x[(ra + 1) * Q1K + j + QT * r]);
  q_fft<false>(a, lds[g], t, j);
  __syncthreads();  // stage 4's reads are done
#pragma unroll
  for (int r = 0; r < 4; ++r) lds[g][q_pad(j + QT * r)] = a[r];
  __syncthreads();
  const long long item = r0 / Q1K;
  const int rl = static_cast<int>(r0 - item * Q1K);
  float4* out = reinterpret_cast<float4*>(halfT + item * QH1 * Q1K + rl);
  for (int e = threadIdx.x; e < 2 * QH1; e += 2 * QT) {
    const int k = e >> 1, h = e & 1;
    const float2 zk = lds[h][q_pad(k)], zm = lds[h][q_pad((Q1K - k) & (Q1K - 1))];
    out[(static_cast<long long>(k) * Q1K >> 1) + h] =
        make_float4(__fmul_rn(0.5f, __fadd_rn(zk.x, zm.x)), __fmul_rn(0.5f, __fsub_rn(zk.y, zm.y)),
                    __fmul_rn(0.5f, __fadd_rn(zk.y, zm.y)), __fmul_rn(0.5f, __fsub_rn(zm.x, zk.x)));
  }
}

// Columns (F0 = 1024) of the transposed half spectrum: forward, times hsT
// (conj for the adjoint), inverse, times 1/1024; one column per workgroup.
__global__ __launch_bounds__(QT) void q1k_cols_kernel(float2* __restrict__ halfT,
                                                      const float2* __restrict__ hsT, int conj_h,
                                                      const float2* __restrict__ tw,
                                                      const int32_t* pred) {
  if (pred_off(pred)) return;
  __shared__ float2 lds[Q_LDS];
  const int j = threadIdx.x;
  const int c = static_cast<int>(blockIdx.x % QH1);
  float2* col = halfT + static_cast<long long>(blockIdx.x) * Q1K;
  const float2* hc = hsT + static_cast<long long>(c) * Q1K;
  QTw t;
  q_twiddles(t, tw, j);
  float2 h[4], a[4];
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const float2 hv = hc[j + QT * r];
    h[r] = conj_h ? conjf2(hv) : hv;
    a[r] = col[j + QT * r];
  }
  q_fft<false>(a, lds, t, j);
#pragma unroll
  for (int r = 0; r < 4; ++r) a[r] = cmul(h[r], a[r]);
  q_fft<true>(a, lds, t, j);
  constexpr float sc = 1.0f / Q1K;
#pragma unroll
  for (int r = 0; r < 4; ++r)
    col[j + QT * r] = make_float2(__fmul_rn(a[r].x, sc), __fmul_rn(a[r].y, sc));
}

// Inverse rows: the transposed half spectra of QR rows -> real rows, times
// 1/1024 (Z[k] = X_a[k] + i X_b[k] and its Hermitian extension, imaginary
// parts of k = 0 and 512 dropped as irfft does).  Loads the transform
// result of thread j of group g into a (pair of rows 2g, 2g + 1).
// Rows r0 .. r0 + QR - 1 (r0 = QR rb) of the half spectrum, inverse
// transformed: a holds the two real rows r0 + 2 g, r0 + 2 g + 1.
__device__ __forceinline__ void q1k_c2r_load(const float2* __restrict__ halfT, float2 (&lds)[2][Q_LDS],
                                             long long rb, const QTw& t, int g, int j,
                                             float2 (&a)[4]) {
  const long long r0 = rb * QR;
  const long long item = r0 / Q1K;
  const int rl = static_cast<int>(r0 - item * Q1K);
  const float4* in = reinterpret_cast<const float4*>(halfT + item * QH1 * Q1K + rl);
  constexpr int nh = Q1K / 2;
  for (int e = threadIdx.x; e < 2 * QH1; e += 2 * QT) {
    const int k = e >> 1, h = e & 1;
    const float4 v = in[(static_cast<long long>(k) * Q1K >> 1) + h];
    float2 aa = make_float2(v.x, v.y), bb = make_float2(v.z, v.w);
    if (k == 0 || k == nh) aa.y = bb.y = 0.0f;
    lds[h][q_pad(k)] = make_float2(__fsub_rn(aa.x, bb.y), __fadd_rn(aa.y, bb.x));
    if (k > 0 && k < nh)
      lds[h][q_pad(Q1K - k)] = make_float2(__fadd_rn(aa.x, bb.y), __fsub_rn(bb.x, aa.y));
  }
  __syncthreads();
#pragma unroll
  for (int r = 0; r < 4; ++r) a[r] = lds[g][q_pad(j + QT * r)];
  q_fft<true>(a, lds[g], t, j);
}

__global__ __launch_bounds__(2 * QT) void q1k_c2r_kernel(const float2* __restrict__ halfT,
                                                         float* __restrict__ y,
                                                         const float2* __restrict__ tw,
                                                         const int32_t* pred) {
  if (pred_off(pred)) return;
  __shared__ float2 lds[2][Q_LDS];
  const int g = threadIdx.x >> 8, j = threadIdx.x & (QT - 1);
  QTw t;
  q_twiddles(t, tw, j);
  float2 a[4];
  const long long rb = q_row_block();
  q1k_c2r_load(halfT, lds, rb, t, g, j, a);
  const long long ra = rb * QR + 2 * g;
  constexpr float sc = 1.0f / Q1K;
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    y[ra * Q1K + j + QT * r] = __fmul_rn(a[r].x, sc);
    y[(ra + 1) * Q1K + j + QT * r] = __fmul_rn(a[r].y, sc);
  }
}

// ---------------------------------- fused AcceleratedPGM gradient step --
//
// For f(x) = 0.5 ||A x - y||^2 with A a real circular convolution over two
// axes (F0, F1), one convolution per iteration serves both the gradient and
// the objective:
//   * G x (G = A^T A: the convolution by |Hs|^2, real on the half grid),
//     and G v = (1 + c) G x - c G x_prev for the extrapolated point
//     v = x + c (x - x_prev) (linearity), so u = v - (1/L) (G v - A^T y);
//   * ||A x - y||^2 = sum_k w_k |Hs[k] X[k] - Y[k]|^2 / (F0 F1) over the
//     half spectrum (Parseval; w_k = 1 on the first and, for even F1, the
//     Nyquist column, 2 elsewhere), X and Y the spectra of x and y.
// Half-grid arrays are F0 x (F1/2 + 1); at 1024 x 1024 they are transposed
// (column k1 contiguous).

// Hermitian part of the (F0, F1) spectrum h at (k0, k1), in float64.
__device__ __forceinline__ double2 hermitian64(const float2* __restrict__ h, int k0, int k1,
                                               int F0, int F1) {
  const float2 a = h[static_cast<long long>(k0) * F1 + k1];
  const float2 b = h[static_cast<long long>((F0 - k0) % F0) * F1 + (F1 - k1) % F1];
  return make_double2(0.5 * (static_cast<double>(a.x) + static_cast<double>(b.x)),
                      0.5 * (static_cast<double>(a.y) - static_cast<double>(b.y)));
}

// Set-up: gs = |Hs|^2 on the half grid, evaluated in float64 from the
// plan's spectrum and rounded once.
__global__ __launch_bounds__(256) void gram_spectrum_kernel(const float2* __restrict__ h,
                                                            float* __restrict__ gs, int F0, int F1,
                                                            int trans) {
  const int H1 = F1 / 2 + 1;
  const long long tot = static_cast<long long>(F0) * H1;
  for (long long e = blockIdx.x * 256ll + threadIdx.x; e < tot; e += 256ll * gridDim.x) {
    const int k0 = static_cast<int>(e / H1), k1 = static_cast<int>(e - static_cast<long long>(k0) * H1);
    const double2 g = hermitian64(h, k0, k1, F0, F1);
    gs[trans ? static_cast<long long>(k1) * F0 + k0 : e] = static_cast<float>(g.x * g.x + g.y * g.y);
  }
}

// Set-up: Yh = rfft2(y) and A^T y in float64, rounded once.  Runs once per
// solve (69 us at 1024 x 1024, 29 of them for A^T y, 21 in float32), one line
// per workgroup in LDS: once, so simple kernels serve.  The rounding of A^T y
// stays in every gradient: in float32, the fused iteration was 6 to 11 % further
// from the float64 one than the iteration with G v had been (512 x 512, 50
// steps: 4.1e-7 against 3.7e-7), with this 3.2e-7.
__global__ __launch_bounds__(256) void twiddle64_kernel(double2* __restrict__ tw, int n) {
  const int k = blockIdx.x * 256 + threadIdx.x;
  if (k >= n) return;
  double sn, cs;
  sincospi(-2.0 * k / n, &sn, &cs);
  tw[k] = make_double2(cs, sn);
}

constexpr int MAXV64 = MAX_POW2 / SH_THREADS;  // values per thread of a line

__global__ __launch_bounds__(SH_THREADS) void rows64_kernel(const float* __restrict__ y,
                                                            double2* __restrict__ half, int n,
                                                            Stages S,
                                                            const double2* __restrict__ tw) {
  extern __shared__ double2 lds64[];
  const int H1 = n / 2 + 1;
  const long long row = blockIdx.x;
  for (int k = threadIdx.x; k < n; k += SH_THREADS)
    lds64[k] = make_double2(static_cast<double>(y[row * n + k]), 0.0);
  __syncthreads();
  mixed<MAXV64>(lds64, n, S, 1, tw, false);
  for (int k = threadIdx.x; k < H1; k += SH_THREADS) half[row * H1 + k] = lds64[k];
}

// Columns: the spectrum of y to out (if not null) and, if h is not null, times
// conj(Hs) and back for A^T y, in place.
__global__ __launch_bounds__(SH_THREADS) void cols64_kernel(double2* __restrict__ half,
                                                            float2* __restrict__ out,
                                                            const float2* __restrict__ h, int n,
                                                            int F1, Stages S,
                                                            const double2* __restrict__ tw,
                                                            int trans) {
  const int H1 = F1 / 2 + 1;
  extern __shared__ double2 lds64[];
  // consecutive columns on one XCD: they share the cache lines of their rows
  int c = blockIdx.x;
  {
    const int G8 = (gridDim.x / 8) * 8;
    if (c < G8) c = (c % 8) * (G8 / 8) + c / 8;
  }
  for (int k = threadIdx.x; k < n; k += SH_THREADS)
    lds64[k] = half[static_cast<long long>(k) * H1 + c];
  __syncthreads();
  mixed<MAXV64>(lds64, n, S, 1, tw, false);
  if (out)
    for (int k = threadIdx.x; k < n; k += SH_THREADS)
      out[trans ? static_cast<long long>(c) * n + k : static_cast<long long>(k) * H1 + c] =
          make_float2(static_cast<float>(lds64[k].x), static_cast<float>(lds64[k].y));
  if (!h) return;
  for (int k = threadIdx.x; k < n; k += SH_THREADS)
    lds64[k] = cmul(conjf2(hermitian64(h, k, c, n, F1)), lds64[k]);
  __syncthreads();
  mixed<MAXV64>(lds64, n, S, 1, tw, true);
  for (int k = threadIdx.x; k < n; k += SH_THREADS)
    half[static_cast<long long>(k) * H1 + c] = lds64[k];
}

// Rows of a half spectrum back to real rows (the imaginary parts of the k = 0
// and, for even n, k = n / 2 bins dropped, as irfft does), times scale.
__global__ __launch_bounds__(SH_THREADS) void rows64_inverse_kernel(
    const double2* __restrict__ half, float* __restrict__ out, int n, Stages S,
    const double2* __restrict__ tw, double scale) {
  extern __shared__ double2 lds64[];
  const int H1 = n / 2 + 1;
  const long long row = blockIdx.x;
  for (int k = threadIdx.x; k < H1; k += SH_THREADS) {
    double2 a = half[row * H1 + k];
    if (k == 0 || 2 * k == n) a.y = 0.0;
    lds64[k] = a;
    if (k > 0 && 2 * k < n) lds64[n - k] = conjf2(a);
  }
  __syncthreads();
  mixed<MAXV64>(lds64, n, S, 1, tw, true);
  for (int k = threadIdx.x; k < n; k += SH_THREADS)
    out[row * n + k] = static_cast<float>(lds64[k].x * scale);
}

// Columns of any length (the 1024-point ones below keep their line in
// registers): forward, objective partial of the workgroup's columns (if
// obj), times gs, inverse, times 1/F0.
template <bool MIXED, int MAXV>
__global__ __launch_bounds__(SH_THREADS) void cols_gram_kernel(
    float2* __restrict__ half, const float2* __restrict__ hs, const float* __restrict__ gs,
    const float2* __restrict__ Yh, double* __restrict__ obj, int n, int log2n, Stages S, int H1,
    int F1, int lpb, const float2* __restrict__ tw, float scale, const int32_t* pred) {
  if (pred_off(pred)) return;
  extern __shared__ float2 lds[];
  __shared__ double sh[4];
  float2* X = lds;
  const int tot = lpb * n;
  const float2* twl = pass_twiddles<MIXED>(X, tot, n, S, tw);
  int blk = blockIdx.x;  // neighbouring columns on one XCD, as in stockham_kernel
  {
    const int G8 = (gridDim.x / 8) * 8;
    if (blk < G8) blk = (blk % 8) * (G8 / 8) + blk / 8;
  }
  const int c0 = blk * lpb, nl = min(lpb, H1 - c0);
  for (int e = threadIdx.x; e < tot; e += SH_THREADS) {
    const int k = e / lpb, l = e - k * lpb;
    X[l * n + k] = l < nl ? half[static_cast<long long>(k) * H1 + c0 + l] : make_float2(0.f, 0.f);
  }
  __syncthreads();
  transform<MIXED, MAXV>(X, n, log2n, S, lpb, twl, false);
  double acc = 0.0;
  for (int e = threadIdx.x; e < tot; e += SH_THREADS) {
    const int k = e / lpb, l = e - k * lpb;
    if (l < nl) {
      const long long o = static_cast<long long>(k) * H1 + c0 + l;
      const float2 a = X[l * n + k];
      if (obj) {
        const float2 p = cmul(hs[o], a), yk = Yh[o];
        const double dx = static_cast<double>(p.x) - static_cast<double>(yk.x);
        const double dy = static_cast<double>(p.y) - static_cast<double>(yk.y);
        const double d = dx * dx + dy * dy;
        acc += (c0 + l == 0 || 2 * (c0 + l) == F1) ? d : 2.0 * d;
      }
      const float g = gs[o];
      X[l * n + k] = make_float2(__fmul_rn(g, a.x), __fmul_rn(g, a.y));
    }
  }
  if (obj) {
    acc = block_sum_f64(acc, sh);
    if (threadIdx.x == 0) obj[blockIdx.x] = acc;
  }
  __syncthreads();
  transform<MIXED, MAXV>(X, n, log2n, S, lpb, twl, true);
  for (int e = threadIdx.x; e < tot; e += SH_THREADS) {
    const int k = e / lpb, l = e - k * lpb;
    if (l < nl) {
      const float2 a = X[l * n + k];
      half[static_cast<long long>(k) * H1 + c0 + l] =
          make_float2(__fmul_rn(a.x, scale), __fmul_rn(a.y, scale));
    }
  }
}

// Columns: forward, objective partial of the column (if obj), times gsT,
// inverse, times 1/1024.
__global__ __launch_bounds__(QT) void q1k_cols_gram_kernel(float2* __restrict__ halfT,
                                                           const float2* __restrict__ hsT,
                                                           const float* __restrict__ gsT,
                                                           const float2* __restrict__ YT,
                                                           double* __restrict__ obj,
                                                           const float2* __restrict__ tw,
                                                           const int32_t* pred) {
  if (pred_off(pred)) return;
  __shared__ float2 lds[Q_LDS];
  __shared__ double sh[4];
  const int j = threadIdx.x;
  const int c = blockIdx.x;
  const long long o = static_cast<long long>(c) * Q1K;
  float2* col = halfT + o;
  QTw t;
  q_twiddles(t, tw, j);
  float g[4];
  float2 h[4], yk[4], a[4];
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    g[r] = gsT[o + j + QT * r];
    if (obj) {
      h[r] = hsT[o + j + QT * r];
      yk[r] = YT[o + j + QT * r];
    }
    a[r] = col[j + QT * r];
  }
  q_fft<false>(a, lds, t, j);
  if (obj) {
    double acc = 0.0;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const float2 p = cmul(h[r], a[r]);
      const double dx = static_cast<double>(p.x) - static_cast<double>(yk[r].x);
      const double dy = static_cast<double>(p.y) - static_cast<double>(yk[r].y);
      acc += dx * dx + dy * dy;
    }
    acc = block_sum_f64(acc, sh);
    if (j == 0) obj[c] = (c == 0 || c == QH1 - 1) ? acc : 2.0 * acc;
  }
#pragma unroll
  for (int r = 0; r < 4; ++r) a[r] = make_float2(__fmul_rn(g[r], a[r].x), __fmul_rn(g[r], a[r].y));
  q_fft<true>(a, lds, t, j);
  constexpr float sc = 1.0f / Q1K;
#pragma unroll
  for (int r = 0; r < 4; ++r)
    col[j + QT * r] = make_float2(__fmul_rn(a[r].x, sc), __fmul_rn(a[r].y, sc));
}

// Statistics of an AcceleratedPGM iteration (apgm_stats_block arguments).
struct ApgmStats {
  const double* obj;
  int nobj;
  double obj_scale;
  const double* tv;
  int ntv;
  double lam;
  const double* res;
  int nres;
  double* hist;
  int32_t* counter;
  int hist_cap;
};

// Inverse rows into G x, then the gradient step:
//   gv = (1 + c) gx_new - c gx_prev,  u = v + b (gv - aty)   (b = -1/L)
// with gx <- gx_new.  With STATS, workgroup 0 reduces the iteration's
// statistics row instead (from partials that the kernels before this one
// on the stream wrote) while workgroups 1 .. Q1K / QR take the row blocks,
// so the row needs no launch of its own.
template <bool STATS>
__global__ __launch_bounds__(2 * QT) void q1k_c2r_step_kernel(
    const float2* __restrict__ halfT, float* __restrict__ gx, const float* __restrict__ v,
    const float* __restrict__ aty, float c1, float c, float b, float* __restrict__ u,
    const float2* __restrict__ tw, ApgmStats st, const int32_t* pred) {
  if (pred_off(pred)) return;
  if (STATS && blockIdx.x == 0) {
    apgm_stats_block<2 * QT>(st.obj, st.nobj, st.obj_scale, st.tv, st.ntv, st.lam, st.res,
                             st.nres, st.hist, st.counter, st.hist_cap);
    return;
  }
  __shared__ float2 lds[2][Q_LDS];
  const int g = threadIdx.x >> 8, j = threadIdx.x & (QT - 1);
  QTw t;
  q_twiddles(t, tw, j);
  float2 a[4];
  const long long rb = q_row_block(STATS ? 1 : 0);
  q1k_c2r_load(halfT, lds, rb, t, g, j, a);
  const long long ra = rb * QR + 2 * g;
  constexpr float sc = 1.0f / Q1K;
#pragma unroll
  for (int r = 0; r < 4; ++r) {
#pragma unroll
    for (int hh = 0; hh < 2; ++hh) {
      const long long e = (ra + hh) * Q1K + j + QT * r;
      const float gn = __fmul_rn(hh ? a[r].y : a[r].x, sc);
      const float gv = __fsub_rn(__fmul_rn(c1, gn), __fmul_rn(c, gx[e]));
      u[e] = __fadd_rn(v[e], __fmul_rn(b, __fsub_rn(gv, aty[e])));
      gx[e] = gn;
    }
  }
}

// The same for rows of any length: workgroup 0 reduces the statistics row if
// STATS, the others take lpb row pairs each.
template <bool MIXED, int MAXV, bool STATS>
__global__ __launch_bounds__(SH_THREADS) void c2r_step_kernel(
    const float2* __restrict__ half, float* __restrict__ gx, const float* __restrict__ v,
    const float* __restrict__ aty, float c1, float c, float b, float* __restrict__ u, int n,
    int log2n, Stages S, long long R, int lpb, const float2* __restrict__ tw, float scale,
    ApgmStats st, const int32_t* pred) {
  if (pred_off(pred)) return;
  if (STATS && blockIdx.x == 0) {
    apgm_stats_block<SH_THREADS>(st.obj, st.nobj, st.obj_scale, st.tv, st.ntv, st.lam, st.res,
                                 st.nres, st.hist, st.counter, st.hist_cap);
    return;
  }
  extern __shared__ float2 lds[];
  float2* X = lds;
  const long long row0 = 2ll * (blockIdx.x - (STATS ? 1 : 0)) * lpb;
  c2r_lines<MIXED, MAXV, false>(half, X, n, log2n, S, RowPairs{R, 0}, lpb, row0 / 2, tw);
  for (int q = threadIdx.x; q < 2 * lpb * n; q += SH_THREADS) {
    const int r = q / n, k = q - r * n;  // real row row0 + r
    if (row0 + r >= R) break;
    const float2 z = X[(r >> 1) * n + k];
    const long long e = (row0 + r) * n + k;
    const float gn = __fmul_rn(r & 1 ? z.y : z.x, scale);
    const float gv = __fsub_rn(__fmul_rn(c1, gn), __fmul_rn(c, gx[e]));
    u[e] = __fadd_rn(v[e], __fmul_rn(b, __fsub_rn(gv, aty[e])));
    gx[e] = gn;
  }
}

// Hermitian part of the (F0, F1) spectrum on the half grid (F0, F1/2 + 1),
// stored transposed (hs[k1 F0 + k0]) if trans.
__global__ __launch_bounds__(256) void hermitian_half_kernel(const float2* __restrict__ h,
                                                             float2* __restrict__ hs, int F0,
                                                             int F1, int trans) {
  const int H1 = F1 / 2 + 1;
  const long long tot = static_cast<long long>(F0) * H1;
  for (long long e = blockIdx.x * 256ll + threadIdx.x; e < tot; e += 256ll * gridDim.x) {
    const int k0 = static_cast<int>(e / H1), k1 = static_cast<int>(e - static_cast<long long>(k0) * H1);
    const float2 a = h[static_cast<long long>(k0) * F1 + k1];
    const int m0 = (F0 - k0) % F0, m1 = (F1 - k1) % F1;
    const float2 b = h[static_cast<long long>(m0) * F1 + m1];
    hs[trans ? static_cast<long long>(k1) * F0 + k0 : e] =
        make_float2(__fmul_rn(0.5f, __fadd_rn(a.x, b.x)), __fmul_rn(0.5f, __fsub_rn(a.y, b.y)));
  }
}

// Elementwise complex product c = a * b (spectrum centring shift).
__global__ __launch_bounds__(256) void cmul_kernel(long long n, const float2* __restrict__ a,
                                                   const float2* __restrict__ b,
                                                   float2* __restrict__ c) {
  for (long long e = blockIdx.x * 256ll + threadIdx.x; e < n; e += 256ll * gridDim.x)
    c[e] = cmul(a[e], b[e]);
}

// ------------------------------------------------------------------ plan --

struct AxisTables {
  int n = 0, log2n = -1;
  Stages st;  // log2n < 0
  float2* tw = nullptr;
};

struct Plan {
  int nd = 0;
  int F[3] = {1, 1, 1};
  long long batch = 1;
  long long fsize = 1;  // product of F
  AxisTables ax[3];
  float2* h = nullptr;     // spectrum (fsize)
  float2* work = nullptr;  // complex workspace (batch * fsize)
  // real 2D path (two axes of 3 or more): Hermitian part of the spectrum on
  // the half grid (F0, F1/2 + 1) and lines per workgroup of the row and column
  // passes
  bool r2c = false;
  float2* hs = nullptr;
  int lpb_rows = 1, lpb_cols = 1;
};

// The 1024 x 1024 real path (transposed half spectrum, 256-thread lines).
bool q1k_path(const Plan& p) { return p.r2c && p.F[0] == Q1K && p.F[1] == Q1K; }

int log2_exact(int n) {
  if (n <= 0 || (n & (n - 1))) return -1;
  int l = 0;
  while ((1 << l) < n) ++l;
  return l;
}

// Stages of a length that is no power of two: primes above 7 first (their
// sums need no twiddle of an earlier stage), then 7, 5 and 3, then the power
// of two in radices 8 and a last 4 or 2.
Stages make_stages(int n) {
  Stages S;
  auto add = [&](int R) { S.R[S.count++] = R; };
  int m = n;
  for (int p = 11; p <= m; p += 2)
    while (m % p == 0 && [&] {
             for (int d = 3; d * d <= p; d += 2)
               if (p % d == 0) return false;
             return true;
           }()) {
      add(p);
      S.twlds = 1;
      m /= p;
    }
  for (int p : {7, 5, 3, 8, 4, 2})
    while (m % p == 0) {
      add(p);
      m /= p;
    }
  auto magic = [](int d) {
    return static_cast<uint32_t>(((1ull << 32) + d - 1) / static_cast<unsigned long long>(d));
  };
  for (int s = 0, Ns = 1; s < S.count; ++s) {
    S.mns[s] = magic(Ns);  // Ns = 1 wraps to 0: the kernels skip it
    S.mnb[s] = magic(n / S.R[s]);
    Ns *= S.R[s];
  }
  return S;
}

// Dynamic LDS of a pass: lpb lines of n values and, for p-term sums, the n
// twiddles.
size_t pass_lds(const AxisTables& t, int lpb) {
  return sizeof(float2) * (static_cast<size_t>(lpb) * t.n + (t.st.twlds ? t.n : 0));
}

// Lines that a workgroup may take: 1024 values, the instances of four values
// a thread (8 x 512 x 512 convolution, 4 lines against 2: 53.7 against 48.2
// us, 8 x 450 x 480 64.3 against 41.3 us); lines longer than that (powers of
// two) 8192.
int line_cap(const AxisTables& t) {
  const int values = t.n <= SH_FEW * SH_THREADS ? SH_FEW * SH_THREADS : 8192;
  return std::max(1, values / t.n);
}

// Whether a pass of l lines of t has an instance that holds them.
bool lines_fit(const AxisTables& t, int l) {
  const int most = t.log2n < 0 ? SH_FEW * SH_THREADS : SH_MAXV * SH_THREADS;
  return l >= 1 && l <= 64 && static_cast<long long>(l) * t.n <= most;
}

// The instance of a pass's kernel for lpb lines of t (see SH_MAXV); mixed
// lengths never take more than 1024 values.
#define SCXR_FFT_KERNEL(K, t, lpb, ...)                            \
  ((t).log2n < 0 ? &K<true, SH_FEW, ##__VA_ARGS__>                 \
   : static_cast<long long>(lpb) * (t).n <= SH_FEW * SH_THREADS    \
       ? &K<false, SH_FEW, ##__VA_ARGS__>                          \
       : &K<false, SH_MAXV, ##__VA_ARGS__>)

int make_tables(AxisTables& t, int n) {
  t.n = n;
  t.log2n = log2_exact(n);
  SCXR_REQUIRE(t.log2n >= 0 ? n <= MAX_POW2 : n <= MAX_DFT, SCXR_ERR_UNSUPPORTED,
               "FFT length %d unsupported (powers of two up to %d, other lengths up to %d)", n,
               MAX_POW2, MAX_DFT);
  if (t.log2n < 0) t.st = make_stages(n);
  const int cnt = n;  // exp(-2 pi i k / n), k < n
  std::vector<float2> tw(cnt);
  for (int k = 0; k < cnt; ++k) {
    const double a = -2.0 * M_PI * static_cast<double>(k) / static_cast<double>(n);
    tw[k] = make_float2(static_cast<float>(std::cos(a)), static_cast<float>(std::sin(a)));
  }
  if (hipMalloc(&t.tw, sizeof(float2) * cnt) != hipSuccess)
    return fail(SCXR_ERR_NOMEM, "hipMalloc of FFT twiddles failed");
  SCXR_HIP(hipMemcpy(t.tw, tw.data(), sizeof(float2) * cnt, hipMemcpyHostToDevice));
  return SCXR_OK;
}

void destroy(Plan& p) {
  for (auto& a : p.ax)
    if (a.tw) (void)hipFree(a.tw), a.tw = nullptr;
  if (p.hs) (void)hipFree(p.hs), p.hs = nullptr;
  if (p.h) (void)hipFree(p.h), p.h = nullptr;
  if (p.work) (void)hipFree(p.work), p.work = nullptr;
}

// One pass along FFT axis a.
int run_pass(const Plan& p, int a, const void* in, void* out, bool in_real, bool out_real,
             bool inverse, bool fused, bool conj_h, const int32_t* pred, hipStream_t s) {
  Pass P{};
  const AxisTables& t = p.ax[a];
  P.n = t.n;
  P.log2n = t.log2n;
  long long stride = 1;
  for (int b = a + 1; b < p.nd; ++b) stride *= p.F[b];
  P.stride = stride;
  P.inner = stride;
  P.lines = p.batch * (p.fsize / t.n);
  // one LDS buffer of lpb lines; lines per workgroup chosen so that a pass
  // has at least ~1024 workgroups
  int lpb = line_cap(t);
  { int q = 1; while (q * 2 <= lpb) q *= 2; lpb = q; }
  while (lpb > 1 && (P.lines + lpb - 1) / lpb < 1024) lpb /= 2;
  lpb = std::min(lpb, 64);
  P.lpb = lpb;
  P.in_real = in_real;
  P.out_real = out_real;
  P.inverse = inverse;
  P.fused = fused;
  P.conj_h = conj_h;
  P.tw = t.tw;
  P.h = p.h;
  const float scale = (inverse || fused) ? 1.0f / static_cast<float>(t.n) : 1.0f;
  const unsigned grid = static_cast<unsigned>((P.lines + lpb - 1) / lpb);
  hipLaunchKernelGGL(SCXR_FFT_KERNEL(stockham_kernel, t, lpb), dim3(grid), dim3(SH_THREADS),
                     pass_lds(t, lpb), s, in, out, P, t.st, scale, pred);
  SCXR_LAUNCHED("fft pass");
  return SCXR_OK;
}

// Row pairs of a plan's images, and their number.
RowPairs row_pairs(const Plan& p) {
  const bool odd = p.batch > 1 && p.F[0] % 2 == 1;
  return {p.batch * p.F[0], odd ? static_cast<unsigned>(p.F[0] + 1) / 2 : 0u};
}
long long pair_count(const Plan& p) { return p.batch * ((p.F[0] + 1) / 2); }

// Real 2D path: rows forward (two real rows per complex FFT), fused column
// pass on the half spectrum, rows inverse.
int convolve_r2c(const Plan& p, const float* x, float* y, bool adj, const int32_t* pred,
                 hipStream_t s) {
  const AxisTables& t1 = p.ax[1];
  const int n = t1.n, H1 = n / 2 + 1;
  const long long R = p.batch * p.F[0];
  float2* half = p.work;  // R rows of H1 (fits in the batch * fsize workspace)
  const RowPairs P1 = row_pairs(p);
  const long long cl = pair_count(p);  // complex row transforms
  if (q1k_path(p)) {
    const unsigned gr = static_cast<unsigned>(R / QR);
    hipLaunchKernelGGL(q1k_r2c_kernel, dim3(gr), dim3(2 * QT), 0, s, x, half, t1.tw, pred);
    SCXR_LAUNCHED("fft r2c rows (1024)");
    hipLaunchKernelGGL(q1k_cols_kernel, dim3(static_cast<unsigned>(p.batch * H1)), dim3(QT), 0, s,
                       half, p.hs, static_cast<int>(adj), p.ax[0].tw, pred);
    SCXR_LAUNCHED("fft half-spectrum columns (1024)");
    hipLaunchKernelGGL(q1k_c2r_kernel, dim3(gr), dim3(2 * QT), 0, s, half, y, t1.tw, pred);
    SCXR_LAUNCHED("fft c2r rows (1024)");
    return SCXR_OK;
  }
  int lr = p.lpb_rows;
  const unsigned gr = static_cast<unsigned>((cl + lr - 1) / lr);
  const size_t lds_r = pass_lds(t1, lr);
  hipLaunchKernelGGL(P1.odd ? SCXR_FFT_KERNEL(r2c_rows_kernel, t1, lr, true)
                            : SCXR_FFT_KERNEL(r2c_rows_kernel, t1, lr, false),
                     dim3(gr), dim3(SH_THREADS), lds_r, s, x, half, n, t1.log2n, t1.st, P1, lr,
                     t1.tw, pred);
  SCXR_LAUNCHED("fft r2c rows");
  // columns of the half spectrum: n0-point transforms at stride H1
  const AxisTables& t0 = p.ax[0];
  Pass P{};
  P.n = t0.n;
  P.log2n = t0.log2n;
  P.stride = H1;
  P.inner = H1;
  P.lines = p.batch * H1;
  P.lpb = p.lpb_cols;
  P.fused = 1;
  P.conj_h = adj;
  P.tw = t0.tw;
  P.h = p.hs;
  const unsigned gc = static_cast<unsigned>((P.lines + P.lpb - 1) / P.lpb);
  hipLaunchKernelGGL(SCXR_FFT_KERNEL(stockham_kernel, t0, P.lpb), dim3(gc), dim3(SH_THREADS),
                     pass_lds(t0, P.lpb), s, static_cast<const void*>(half),
                     static_cast<void*>(half), P, t0.st, 1.0f / static_cast<float>(t0.n), pred);
  SCXR_LAUNCHED("fft half-spectrum columns");
  hipLaunchKernelGGL(P1.odd ? SCXR_FFT_KERNEL(c2r_rows_kernel, t1, lr, true)
                            : SCXR_FFT_KERNEL(c2r_rows_kernel, t1, lr, false),
                     dim3(gr), dim3(SH_THREADS), lds_r, s, half, y, n, t1.log2n, t1.st, P1, lr,
                     t1.tw, 1.0f / static_cast<float>(n), pred);
  SCXR_LAUNCHED("fft c2r rows");
  return SCXR_OK;
}

// y = real(ifftn(H' * fftn(x))) with H' = H or conj(H).
int convolve(const Plan& p, const float* x, float* y, bool adj, const int32_t* pred,
             hipStream_t s) {
  if (p.r2c) return convolve_r2c(p, x, y, adj, pred, s);
  if (p.nd == 1) return run_pass(p, 0, x, y, true, true, false, true, adj, pred, s);
  int rc;
  // forward along F{d-1} .. F1 (first pass reads the real input)
  for (int a = p.nd - 1, first = 1; a >= 1; --a, first = 0) {
    rc = run_pass(p, a, first ? static_cast<const void*>(x) : p.work, p.work, first, false, false,
                  false, false, pred, s);
    if (rc) return rc;
  }
  rc = run_pass(p, 0, p.work, p.work, false, false, false, true, adj, pred, s);
  if (rc) return rc;
  for (int a = 1; a < p.nd; ++a) {
    const bool last = (a == p.nd - 1);
    rc = run_pass(p, a, p.work, last ? static_cast<void*>(y) : p.work, false, last, true, false,
                  false, pred, s);
    if (rc) return rc;
  }
  return SCXR_OK;
}

// Complex fftn / ifftn of x (complex or real input) into out (complex).
int fftn(const Plan& p, const void* x, bool x_real, float2* out, bool inverse, const int32_t* pred,
         hipStream_t s) {
  for (int a = p.nd - 1, first = 1; a >= 0; --a, first = 0) {
    const int rc = run_pass(p, a, first ? x : static_cast<const void*>(out), out,
                            first && x_real, false, inverse, false, false, pred, s);
    if (rc) return rc;
  }
  return SCXR_OK;
}

}  // namespace fft
}  // namespace scxr

struct scxr_cconv_plan {
  scxr::fft::Plan p;
};

using namespace scxr::fft;

extern "C" {

int scxr_cconv_plan_create(int32_t ndim, const int32_t* fshape, int64_t batch,
                           scxr_cconv_plan** out) {
  SCXR_REQUIRE(out && fshape && ndim >= 1 && ndim <= 3 && batch >= 1, SCXR_ERR_ARG,
               "bad cconv plan arguments");
  auto* plan = new scxr_cconv_plan();
  Plan& p = plan->p;
  p.nd = ndim;
  p.batch = batch;
  p.fsize = 1;
  int rc = SCXR_OK;
  for (int a = 0; a < ndim && rc == SCXR_OK; ++a) {
    if (fshape[a] < 1) rc = fail(SCXR_ERR_SHAPE, "non-positive FFT length");
    if (rc == SCXR_OK) {
      p.F[a] = fshape[a];
      p.fsize *= fshape[a];
      rc = make_tables(p.ax[a], fshape[a]);
    }
  }
  if (rc == SCXR_OK && hipMalloc(&p.h, sizeof(float2) * p.fsize) != hipSuccess)
    rc = fail(SCXR_ERR_NOMEM, "hipMalloc of the spectrum failed");
  if (rc == SCXR_OK && hipMalloc(&p.work, sizeof(float2) * p.fsize * p.batch) != hipSuccess)
    rc = fail(SCXR_ERR_NOMEM, "hipMalloc of the FFT workspace failed");
  if (rc == SCXR_OK && ndim == 2 && p.F[0] > 2 && p.F[1] > 2) {
    p.r2c = true;
    const long long H1 = p.F[1] / 2 + 1;
    if (hipMalloc(&p.hs, sizeof(float2) * p.F[0] * H1) != hipSuccess)
      rc = fail(SCXR_ERR_NOMEM, "hipMalloc of the half spectrum failed");
    // lines per workgroup: as many as line_cap allows (at most the 64 lines
    // that a column pass tabulates) while the pass keeps at least 512
    // workgroups (SCXR_FFT_LPB="rows,cols" overrides)
    auto pick = [](long long lines, const AxisTables& t) {
      int l = std::min(64, line_cap(t));
      while (l > 1 && (lines + l - 1) / l < 512) l /= 2;
      return l;
    };
    p.lpb_rows = pick(pair_count(p), p.ax[1]);
    p.lpb_cols = pick(p.batch * H1, p.ax[0]);
    if (const char* env = std::getenv("SCXR_FFT_LPB")) {
      int a = 0, b = 0;
      if (std::sscanf(env, "%d,%d", &a, &b) == 2 && lines_fit(p.ax[1], a) &&
          lines_fit(p.ax[0], b)) {
        p.lpb_rows = a;
        p.lpb_cols = b;
      }
    }
  }
  if (rc != SCXR_OK) {
    destroy(p);
    delete plan;
    return rc;
  }
  *out = plan;
  return SCXR_OK;
}

int scxr_cconv_plan_destroy(scxr_cconv_plan* plan) {
  if (!plan) return SCXR_OK;
  destroy(plan->p);
  delete plan;
  return SCXR_OK;
}

int scxr_cconv_set_spectrum(scxr_cconv_plan* plan, const float* h, int32_t h_is_dft,
                            const float* shift, void* stream) {
  SCXR_REQUIRE(plan && h, SCXR_ERR_ARG, "null argument to cconv_set_spectrum");
  Plan& p = plan->p;
  const hipStream_t s = as_stream(stream);
  if (h_is_dft) {
    SCXR_HIP(hipMemcpyAsync(p.h, h, sizeof(float2) * p.fsize, hipMemcpyDeviceToDevice, s));
  } else {
    // h: real, zero-padded to the FFT shape (batch 1)
    Plan q = p;
    q.batch = 1;
    const int rc = fftn(q, h, true, p.h, false, nullptr, s);
    if (rc) return rc;
  }
  if (shift) {
    hipLaunchKernelGGL(cmul_kernel, dim3(256), dim3(256), 0, s, p.fsize, p.h,
                       reinterpret_cast<const float2*>(shift), p.h);
    SCXR_LAUNCHED("cconv shift");
  }
  if (p.r2c) {
    hipLaunchKernelGGL(hermitian_half_kernel, dim3(256), dim3(256), 0, s, p.h, p.hs, p.F[0],
                       p.F[1], static_cast<int>(q1k_path(p)));
    SCXR_LAUNCHED("cconv half spectrum");
  }
  return SCXR_OK;
}

int scxr_cconv_spectrum(const scxr_cconv_plan* plan, float* out, void* stream) {
  SCXR_REQUIRE(plan && out, SCXR_ERR_ARG, "null argument to cconv_spectrum");
  SCXR_HIP(hipMemcpyAsync(out, plan->p.h, sizeof(float2) * plan->p.fsize,
                          hipMemcpyDeviceToDevice, as_stream(stream)));
  return SCXR_OK;
}

int scxr_cconv_apply(const scxr_cconv_plan* plan, const float* x, float* y, int32_t adjoint,
                     const int32_t* pred, void* stream) {
  SCXR_REQUIRE(plan && x && y, SCXR_ERR_ARG, "null argument to cconv_apply");
  return convolve(plan->p, x, y, adjoint != 0, pred, as_stream(stream));
}

}  // extern "C"

// Workgroups of the fused gradient step's column pass, one objective partial
// each (0: the plan is not one real two-axis convolution).
static int apgm_parts(const Plan& p) {
  if (!p.r2c || p.batch != 1) return 0;
  const int H1 = p.F[1] / 2 + 1;
  return q1k_path(p) ? H1 : static_cast<int>(ceil_div(H1, p.lpb_cols));
}

// The three kernels of one fused gradient step; st (nullable) adds the
// statistics row to the last of them.
static int apgm_grad(const scxr_cconv_plan* plan, const float* x, const float* gs,
                     const float* Yh, double* obj, float* gx, const float* v, const float* aty,
                     float c, float b, float* u, const ApgmStats* st, const int32_t* pred,
                     hipStream_t s) {
  SCXR_REQUIRE(plan && x && gs && gx && v && aty && u && (!obj || Yh), SCXR_ERR_ARG,
               "null argument to cconv_apgm_grad");
  const Plan& p = plan->p;
  SCXR_REQUIRE(apgm_parts(p) > 0, SCXR_ERR_UNSUPPORTED,
               "fused APGM gradient needs a plan of one real two-axis convolution");
  float2* half = p.work;
  if (!q1k_path(p)) {
    const AxisTables &t0 = p.ax[0], &t1 = p.ax[1];
    const int n0 = t0.n, n1 = t1.n, H1 = n1 / 2 + 1, lr = p.lpb_rows;
    const unsigned gr = ceil_div((n0 + 1) / 2, lr);
    hipLaunchKernelGGL(SCXR_FFT_KERNEL(r2c_rows_kernel, t1, lr, false), dim3(gr), dim3(SH_THREADS),
                       pass_lds(t1, lr), s, x, half, n1, t1.log2n, t1.st,
                       row_pairs(p), lr, t1.tw, pred);
    SCXR_LAUNCHED("fft r2c rows");
    hipLaunchKernelGGL(SCXR_FFT_KERNEL(cols_gram_kernel, t0, p.lpb_cols),
                       dim3(apgm_parts(p)), dim3(SH_THREADS), pass_lds(t0, p.lpb_cols), s, half,
                       p.hs, gs, reinterpret_cast<const float2*>(Yh), obj, n0, t0.log2n, t0.st, H1,
                       n1, p.lpb_cols, t0.tw, 1.0f / static_cast<float>(n0), pred);
    SCXR_LAUNCHED("fft gram columns");
    const float sc = 1.0f / static_cast<float>(n1);
    if (st)
      hipLaunchKernelGGL(SCXR_FFT_KERNEL(c2r_step_kernel, t1, lr, true),
                         dim3(gr + 1), dim3(SH_THREADS), pass_lds(t1, lr), s, half, gx, v, aty,
                         1.0f + c, c, b, u, n1, t1.log2n, t1.st, static_cast<long long>(n0), lr,
                         t1.tw, sc, *st, pred);
    else
      hipLaunchKernelGGL(SCXR_FFT_KERNEL(c2r_step_kernel, t1, lr, false),
                         dim3(gr), dim3(SH_THREADS), pass_lds(t1, lr), s, half, gx, v, aty,
                         1.0f + c, c, b, u, n1, t1.log2n, t1.st, static_cast<long long>(n0), lr,
                         t1.tw, sc, ApgmStats{}, pred);
    SCXR_LAUNCHED("fft c2r gradient step");
    return SCXR_OK;
  }
  constexpr int H1 = Q1K / 2 + 1;
  hipLaunchKernelGGL(q1k_r2c_kernel, dim3(Q1K / QR), dim3(2 * QT), 0, s, x, half, p.ax[1].tw,
                     pred);
  SCXR_LAUNCHED("fft r2c rows (1024)");
  hipLaunchKernelGGL(q1k_cols_gram_kernel, dim3(H1), dim3(QT), 0, s, half, p.hs, gs,
                     reinterpret_cast<const float2*>(Yh), obj, p.ax[0].tw, pred);
  SCXR_LAUNCHED("fft gram columns (1024)");
  if (st) {
    hipLaunchKernelGGL(q1k_c2r_step_kernel<true>, dim3(Q1K / QR + 1), dim3(2 * QT), 0, s, half,
                       gx, v, aty, 1.0f + c, c, b, u, p.ax[1].tw, *st, pred);
    SCXR_LAUNCHED("fft c2r gradient step + statistics row (1024)");
  } else {
    hipLaunchKernelGGL(q1k_c2r_step_kernel<false>, dim3(Q1K / QR), dim3(2 * QT), 0, s, half, gx,
                       v, aty, 1.0f + c, c, b, u, p.ax[1].tw, ApgmStats{}, pred);
    SCXR_LAUNCHED("fft c2r gradient step (1024)");
  }
  return SCXR_OK;
}

extern "C" {

int32_t scxr_cconv_apgm_parts(const scxr_cconv_plan* plan) {
  return plan ? apgm_parts(plan->p) : 0;
}

int64_t scxr_cconv_apgm_setup_ws(const scxr_cconv_plan* plan) {
  if (!plan || apgm_parts(plan->p) <= 0) return 0;
  const Plan& p = plan->p;
  return 2 * (static_cast<int64_t>(p.F[0]) * (p.F[1] / 2 + 1) + p.F[0] + p.F[1]);
}

int scxr_cconv_apgm_setup(const scxr_cconv_plan* plan, const float* y, float* gs, float* Yh,
                          double* ws, void* stream) {
  SCXR_REQUIRE(gs && Yh, SCXR_ERR_ARG, "null argument to cconv_apgm_setup");
  return scxr_cconv_apgm_setup_aty(plan, y, gs, Yh, nullptr, ws, stream);
}

int scxr_cconv_apgm_setup_aty(const scxr_cconv_plan* plan, const float* y, float* gs, float* Yh,
                              float* aty, double* ws, void* stream) {
  SCXR_REQUIRE(plan && y && ws && (aty || (gs && Yh)), SCXR_ERR_ARG,
               "null argument to cconv_apgm_setup");
  const Plan& p = plan->p;
  SCXR_REQUIRE(apgm_parts(p) > 0, SCXR_ERR_UNSUPPORTED,
               "fused APGM set-up needs a plan of one real two-axis convolution");
  const hipStream_t s = as_stream(stream);
  const int n0 = p.F[0], n1 = p.F[1], H1 = n1 / 2 + 1, trans = q1k_path(p);
  double2* half = reinterpret_cast<double2*>(ws);
  double2* tw0 = half + static_cast<long long>(n0) * H1;
  double2* tw1 = tw0 + n0;
  if (gs) {
    hipLaunchKernelGGL(gram_spectrum_kernel, dim3(1024), dim3(256), 0, s, p.h, gs, n0, n1, trans);
    SCXR_LAUNCHED("cconv gram spectrum");
  }
  hipLaunchKernelGGL(twiddle64_kernel, dim3(ceil_div(n0, 256)), dim3(256), 0, s, tw0, n0);
  SCXR_LAUNCHED("cconv twiddles");
  hipLaunchKernelGGL(twiddle64_kernel, dim3(ceil_div(n1, 256)), dim3(256), 0, s, tw1, n1);
  SCXR_LAUNCHED("cconv twiddles");
  hipLaunchKernelGGL(rows64_kernel, dim3(n0), dim3(SH_THREADS), sizeof(double2) * n1, s, y, half,
                     n1, make_stages(n1), tw1);
  SCXR_LAUNCHED("cconv float64 rows");
  hipLaunchKernelGGL(cols64_kernel, dim3(H1), dim3(SH_THREADS), sizeof(double2) * n0, s, half,
                     reinterpret_cast<float2*>(Yh), aty ? p.h : nullptr, n0, n1, make_stages(n0),
                     tw0, trans);
  SCXR_LAUNCHED("cconv float64 columns");
  if (aty) {
    hipLaunchKernelGGL(rows64_inverse_kernel, dim3(n0), dim3(SH_THREADS), sizeof(double2) * n1, s,
                       half, aty, n1, make_stages(n1), tw1, 1.0 / (static_cast<double>(n0) * n1));
    SCXR_LAUNCHED("cconv float64 inverse rows");
  }
  return SCXR_OK;
}

int scxr_cconv_apgm_grad(const scxr_cconv_plan* plan, const float* x, const float* gs,
                         const float* Yh, double* obj, float* gx, const float* v,
                         const float* aty, float c, float b, float* u, const int32_t* pred,
                         void* stream) {
  return apgm_grad(plan, x, gs, Yh, obj, gx, v, aty, c, b, u, nullptr, pred, as_stream(stream));
}

int scxr_cconv_apgm_grad_itstat(const scxr_cconv_plan* plan, const float* x, const float* gs,
                                const float* Yh, double* obj, float* gx, const float* v,
                                const float* aty, float c, float b, float* u, double obj_scale,
                                const double* tv, int32_t ntv, double lam, const double* res,
                                int32_t nres, double* hist, int32_t* counter, int32_t hist_cap,
                                const int32_t* pred, void* stream) {
  SCXR_REQUIRE(obj && Yh && tv && res && hist && counter && ntv > 0 && nres > 0 && hist_cap > 0,
               SCXR_ERR_ARG, "bad cconv_apgm_grad_itstat arguments");
  SCXR_REQUIRE(plan, SCXR_ERR_ARG, "null argument to cconv_apgm_grad");
  const ApgmStats st{obj, apgm_parts(plan->p), obj_scale, tv, ntv, lam, res, nres, hist, counter,
                     hist_cap};
  return apgm_grad(plan, x, gs, Yh, obj, gx, v, aty, c, b, u, &st, pred, as_stream(stream));
}

int scxr_fftn(const scxr_cconv_plan* plan, const float* x, int32_t x_real, float* out,
              int32_t inverse, const int32_t* pred, void* stream) {
  SCXR_REQUIRE(plan && x && out, SCXR_ERR_ARG, "null argument to fftn");
  return fftn(plan->p, x, x_real != 0, reinterpret_cast<float2*>(out), inverse != 0, pred,
              as_stream(stream));
}

}  // extern "C"
