// One-dimensional complex FP32 transforms of mixed radix in LDS, the passes of the centred facet FFTs.
//
// A transform of n points runs in place in LDS by decimation in frequency: the stage of radix r over
// sub-transforms of L = r m points reads x[j + i m] (i < r), forms their r-point DFT, multiplies
// output k by exp(-2 pi i j k / L) and writes it back to j + k m, so no stage needs a second buffer
// and a stage's butterflies are independent.  After the last stage frequency
// k = k1 + r1 (k2 + r2 (k3 + ...)) lies at k1 m1 + k2 m2 + ..., which the store looks up (`perm`).
// Odd radices use the symmetry of their DFT matrix ((r - 1)^2 multiplications of a real by a
// complex value instead of r^2 complex ones).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

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
  float c[R], s[R];
  constexpr FftTable() : c(), s() {
    for (int k = 0; k < R; ++k) {
      c[k] = float(fft_cos(k, R));
      s[k] = float(fft_sin(k, R));
    }
  }
};

__device__ __forceinline__ float2 fft_add(float2 a, float2 b) { return make_float2(a.x + b.x, a.y + b.y); }
__device__ __forceinline__ float2 fft_sub(float2 a, float2 b) { return make_float2(a.x - b.x, a.y - b.y); }
__device__ __forceinline__ float2 fft_mul(float2 a, float2 w) {
  return make_float2(fmaf(a.x, w.x, -a.y * w.y), fmaf(a.x, w.y, a.y * w.x));
}
__device__ __forceinline__ float2 fft_mi(float2 a) { return make_float2(a.y, -a.x); }  // -i a

// x <- its R-point DFT (forward sign)
template <int R>
__device__ __forceinline__ void fft_dft(float2 (&x)[R]) {
  if constexpr (R == 2) {
    const float2 a = x[0];
    x[0] = fft_add(a, x[1]);
    x[1] = fft_sub(a, x[1]);
  } else if constexpr (R == 4) {
    const float2 a = fft_add(x[0], x[2]), b = fft_sub(x[0], x[2]), c = fft_add(x[1], x[3]), d = fft_mi(fft_sub(x[1], x[3]));
    x[0] = fft_add(a, c);
    x[1] = fft_add(b, d);
    x[2] = fft_sub(a, c);
    x[3] = fft_sub(b, d);
  } else if constexpr (R == 8) {
    float2 e[4] = {x[0], x[2], x[4], x[6]}, o[4] = {x[1], x[3], x[5], x[7]};
    fft_dft<4>(e);
    fft_dft<4>(o);
    constexpr float h = float(fft_cos(1, 8));
    o[1] = make_float2(h * (o[1].x + o[1].y), h * (o[1].y - o[1].x));
    o[2] = fft_mi(o[2]);
    o[3] = make_float2(h * (o[3].y - o[3].x), -h * (o[3].x + o[3].y));
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      x[k] = fft_add(e[k], o[k]);
      x[k + 4] = fft_sub(e[k], o[k]);
    }
  } else {
    constexpr FftTable<R> T;
    constexpr int H = (R - 1) / 2;
    float2 p[H], q[H];
    float2 sum = x[0];
#pragma unroll
    for (int j = 0; j < H; ++j) {
      p[j] = fft_add(x[j + 1], x[R - 1 - j]);
      q[j] = fft_sub(x[j + 1], x[R - 1 - j]);
      sum = fft_add(sum, p[j]);
    }
    const float2 x0 = x[0];
    x[0] = sum;
#pragma unroll
    for (int k = 1; k <= H; ++k) {
      float2 a = x0, b = make_float2(0.f, 0.f);
#pragma unroll
      for (int j = 0; j < H; ++j) {
        const float c = T.c[(k * (j + 1)) % R], s = T.s[(k * (j + 1)) % R];
        a.x = fmaf(p[j].x, c, a.x);
        a.y = fmaf(p[j].y, c, a.y);
        b.x = fmaf(q[j].x, s, b.x);
        b.y = fmaf(q[j].y, s, b.y);
      }
      x[k] = make_float2(a.x + b.y, a.y - b.x);      // a - i b
      x[R - k] = make_float2(a.x - b.y, a.y + b.x);  // a + i b
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
    float2 x[R];
#pragma unroll
    for (int k = 0; k < R; ++k) x[k] = b[k * off];
    fft_dft<R>(x);
    if (!last) {
      const float2* w = tw;
      const int ws = __mul24(j, step);
#pragma unroll
      for (int k = 1; k < R; ++k) {
        w += ws;
        x[k] = fft_mul(x[k], *w);
      }
    }
#pragma unroll
    for (int k = 0; k < R; ++k) b[k * off] = x[k];
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
