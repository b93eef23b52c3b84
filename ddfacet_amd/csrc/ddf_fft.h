// One-dimensional complex transforms of mixed radix in LDS, the passes of the centred facet FFTs.  Values are
// stored in FP32.
//
// A transform of n points runs in place in LDS by decimation in frequency: the stage of radix r over
// sub-transforms of L = r m points reads x[j + i m] (i < r), forms their r-point DFT, multiplies
// output k by exp(-2 pi i j k / L) and writes it back to j + k m, so no stage needs a second buffer
// and a stage's butterflies are independent.  After the last stage frequency
// k = k1 + r1 (k2 + r2 (k3 + ...)) lies at k1 m1 + k2 m2 + ..., which the store looks up (`perm`).
// Odd radices use the symmetry of their DFT matrix ((r - 1)^2 multiplications of a real by a
// complex value instead of r^2 complex ones).
//
// A butterfly of up to 8 points and its twiddle products are FP64, rounded once when a value is stored: with FP32
// butterflies a stage rounds five times over, and the factors' constants, rounded to FP32, scale the whole
// result by up to 9e-8.  Relative L2 error of the 2-D transform at 225, 243, 405, 512, 675 points: FP32 butterflies
// 1.2, 1.3, 1.4, 1.4, 1.5e-7, rocFFT 1.1, 1.2, 1.4, 1.2, 1.4e-7, these 0.7, 0.9, 1.0, 0.7,
// 1.0e-7.  484 planes of 975^2: columns 3.0 ms, rows 2.5 (2.8 and 2.1 with FP32 butterflies).
// Radices 11 and 13 are FP32 with their constants in two parts, and no further from 64 bits than rocFFT at
// lengths that have them; FP64 would take 118 registers a lane in place of 71.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>

namespace ddf {

constexpr int kFftStages = 14;

// The factorisation of a length and the tables made for it on the device.
struct FftDims {
  int n, nst;
  int radix[kFftStages];
  int m[kFftStages];            // points between the inputs of a butterfly of the stage
  uint32_t rcp_m[kFftStages];   // ceil(2^32 / m): t / m = mulhi(t, rcp_m) for t < 2^16, m > 1
  uint32_t rcp_b[kFftStages];   // the same for n / radix (butterflies of one transform)
  uint32_t rcp_n;
  const float2* tw;             // [n] exp(-2 pi i k / n)
  const uint16_t* perm;         // [n] place of frequency k after the last stage
};

// t / d by its reciprocal rcp = ceil(2^32 / d): exact for t d < 2^32 (t and d here below 2^16)
__device__ __forceinline__ int fft_div(int t, int d, uint32_t rcp) { return d == 1 ? t : int(__umulhi(uint32_t(t), rcp)); }

// cos and sin of 2 pi a / b at compile time, by their Taylor series after reduction to an octant
constexpr double fft_taylor(double x, bool cosine) {
  double term = cosine ? 1.0 : x, sum = term;
  for (int k = cosine ? 1 : 2; k < 40; k += 2) {
    term *= -x * x / double(k * (k + 1));
    sum += term;
  }
  return sum;
}
constexpr double fft_cos(int a, int b);
constexpr double fft_sin(int a, int b) {
  const double pi = 3.14159265358979323846264338327950288;
  a %= b;
  if (2 * a > b) return -fft_sin(b - a, b);
  if (4 * a > b) return fft_sin(b - 2 * a, 2 * b);  // sin(pi - x)
  if (8 * a > b) return fft_cos(b - 4 * a, 4 * b);  // cos(pi/2 - x)
  return fft_taylor(2 * pi * a / b, false);
}
constexpr double fft_cos(int a, int b) {
  const double pi = 3.14159265358979323846264338327950288;
  a %= b;
  if (2 * a > b) return fft_cos(b - a, b);
  if (4 * a > b) return -fft_cos(b - 2 * a, 2 * b);
  if (8 * a > b) return fft_sin(b - 4 * a, 4 * b);
  return fft_taylor(2 * pi * a / b, true);
}

template <int R>
struct FftTable {
  double c[R], s[R];
  constexpr FftTable() : c(), s() {
    for (int k = 0; k < R; ++k) {
      c[k] = fft_cos(k, R);
      s[k] = fft_sin(k, R);
    }
  }
};

struct FftD2 {
  double x, y;
};
template <typename V>
__device__ __forceinline__ V fft_add(V a, V b) { return V{a.x + b.x, a.y + b.y}; }
template <typename V>
__device__ __forceinline__ V fft_sub(V a, V b) { return V{a.x - b.x, a.y - b.y}; }
template <typename V>
__device__ __forceinline__ V fft_mi(V a) { return V{a.y, -a.x}; }  // -i a
// a + p c: FP32 takes what the constant's first part leaves over first
__device__ __forceinline__ double fft_mac(double a, double p, double c) { return fma(p, c, a); }
__device__ __forceinline__ float fft_mac(float a, float p, double c) {
  return fmaf(p, float(c), fmaf(p, float(c - double(float(c))), a));
}

// x <- its R-point DFT (forward sign)
template <int R, typename V>
__device__ __forceinline__ void fft_dft(V (&x)[R]) {
  using T = decltype(V::x);
  if constexpr (R == 2) {
    const V a = x[0];
    x[0] = fft_add(a, x[1]);
    x[1] = fft_sub(a, x[1]);
  } else if constexpr (R == 4) {
    const V a = fft_add(x[0], x[2]), b = fft_sub(x[0], x[2]), c = fft_add(x[1], x[3]), d = fft_mi(fft_sub(x[1], x[3]));
    x[0] = fft_add(a, c);
    x[1] = fft_add(b, d);
    x[2] = fft_sub(a, c);
    x[3] = fft_sub(b, d);
  } else if constexpr (R == 8) {
    V e[4] = {x[0], x[2], x[4], x[6]}, o[4] = {x[1], x[3], x[5], x[7]};
    fft_dft<4>(e);
    fft_dft<4>(o);
    constexpr T h = T(fft_cos(1, 8));
    o[1] = V{h * (o[1].x + o[1].y), h * (o[1].y - o[1].x)};
    o[2] = fft_mi(o[2]);
    o[3] = V{h * (o[3].y - o[3].x), -h * (o[3].x + o[3].y)};
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      x[k] = fft_add(e[k], o[k]);
      x[k + 4] = fft_sub(e[k], o[k]);
    }
  } else {
    constexpr FftTable<R> tab;
    constexpr int H = (R - 1) / 2;
    V p[H], q[H];
    V sum = x[0];
#pragma unroll
    for (int j = 0; j < H; ++j) {
      p[j] = fft_add(x[j + 1], x[R - 1 - j]);
      q[j] = fft_sub(x[j + 1], x[R - 1 - j]);
      sum = fft_add(sum, p[j]);
    }
    const V x0 = x[0];
    x[0] = sum;
#pragma unroll
    for (int k = 1; k <= H; ++k) {
      V a = x0, b = V{T(0), T(0)};
#pragma unroll
      for (int j = 0; j < H; ++j) {
        const double c = tab.c[(k * (j + 1)) % R], s = tab.s[(k * (j + 1)) % R];
        a = V{fft_mac(a.x, p[j].x, c), fft_mac(a.y, p[j].y, c)};
        b = V{fft_mac(b.x, q[j].x, s), fft_mac(b.y, q[j].y, s)};
      }
      x[k] = V{a.x + b.y, a.y - b.x};      // a - i b
      x[R - k] = V{a.x - b.y, a.y + b.x};  // a + i b
    }
  }
}

// One stage of `count` transforms in LDS: point i of transform t at buf[t pt + i pi].  TFAST: the
// transforms vary fastest over the threads (a power of two of them: columns side by side), else the
// butterflies of one transform do (rows).
template <int R, bool TFAST>
__device__ __forceinline__ void fft_stage(float2* buf, const float2* tw, const FftDims& d, int s, int count, int log_count,
                                          int pt, int pi) {
  const int m = d.m[s], nb = d.n / R, L = m * R, step = d.n / L, off = m * pi;
  const bool last = m == 1;
  for (int i = threadIdx.x; i < nb * count; i += blockDim.x) {
    int t, u;
    if (TFAST) {
      t = i & (count - 1);
      u = i >> log_count;
    } else {
      t = fft_div(i, nb, d.rcp_b[s]);
      u = i - __mul24(t, nb);
    }
    // (24-bit products: a full 32-bit one takes four times as long)
    const int q = fft_div(u, m, d.rcp_m[s]), j = u - __mul24(q, m);
    float2* b = buf + (__mul24(t, pt) + __mul24(__mul24(q, L) + j, pi));
    using V = typename std::conditional<(R <= 8), FftD2, float2>::type;
    using S = decltype(V::x);
    V x[R];
#pragma unroll
    for (int k = 0; k < R; ++k) x[k] = V{S(b[k * off].x), S(b[k * off].y)};
    fft_dft<R>(x);
    if (!last) {
      const float2* w = tw;
      const int ws = __mul24(j, step);
#pragma unroll
      for (int k = 1; k < R; ++k) {
        w += ws;
        const FftD2 v = {double(x[k].x), double(x[k].y)}, tw_k = {double(w->x), double(w->y)};
        x[k] = V{S(fma(v.x, tw_k.x, -v.y * tw_k.y)), S(fma(v.x, tw_k.y, v.y * tw_k.x))};
      }
    }
#pragma unroll
    for (int k = 0; k < R; ++k) b[k * off] = make_float2(float(x[k].x), float(x[k].y));
  }
}

template <bool TFAST>
__device__ __forceinline__ void fft_stages(float2* buf, const float2* tw, const FftDims& d, int count, int log_count, int pt,
                                           int pi) {
  for (int s = 0; s < d.nst; ++s) {
    switch (d.radix[s]) {
      case 2: fft_stage<2, TFAST>(buf, tw, d, s, count, log_count, pt, pi); break;
      case 3: fft_stage<3, TFAST>(buf, tw, d, s, count, log_count, pt, pi); break;
      case 4: fft_stage<4, TFAST>(buf, tw, d, s, count, log_count, pt, pi); break;
      case 5: fft_stage<5, TFAST>(buf, tw, d, s, count, log_count, pt, pi); break;
      case 7: fft_stage<7, TFAST>(buf, tw, d, s, count, log_count, pt, pi); break;
      case 8: fft_stage<8, TFAST>(buf, tw, d, s, count, log_count, pt, pi); break;
      case 11: fft_stage<11, TFAST>(buf, tw, d, s, count, log_count, pt, pi); break;
      case 13: fft_stage<13, TFAST>(buf, tw, d, s, count, log_count, pt, pi); break;
    }
    __syncthreads();
  }
}

}  // namespace ddf
