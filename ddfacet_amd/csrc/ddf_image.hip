// Facet image side of the major cycle on gfx950: centred facet FFTs (ddf_fft.h; rocFFT for lengths
// outside its factors or its LDS and for the facet models), the facet normalisation image, the facet stitch and the model-to-facet extraction.
//
//   ddf_fft2c          ModFFTW.FFTW_2Donly.fft / .ifft (DDFacet/ToolsDir/ModFFTW.py:557-600):
//                      forward  A <- fftshift(fft2(ifftshift(A))) / N^2,
//                      inverse  A <- fftshift(ifft2(ifftshift(A))) * N^2 (unnormalised),
//                      both times `scale` (GridToIm's OverS^2, ClassDDEGridMachine.py:1186-1190).
//   ddf_facet_norm     BuildFacetNormImage (ClassFacetMachine.py:1289-1325): sum of the facets'
//                      spatial weights on the main image, facets added in index order.
//   ddf_stitch         FacetsToIm_Channel, kind Dirty / PSF (ClassFacetMachine.py:1331-1416).
//   ddf_model_to_grid  GiveModelTessel(ToGrid=False, ApplyNorm=True) (ClassImToGrid.py:138-264)
//                      followed by the forward FFT of get(TranformModelInput="FT")
//                      (ClassDDEGridMachine.py:951-958).
// The stitch, the norm image and the cut's adjoint are gathers over main-image pixels that add the
// covering facets in facet order: no atomics, and the FP32 sums are formed in the reference's order.
#include <hip/hip_runtime.h>
#include <rocfft/rocfft.h>

#include <algorithm>
#include <cmath>
#include <map>
#include <mutex>
#include <string>
#include <tuple>
#include <type_traits>
#include <utility>
#include <vector>

#include "../../include/ddfgpu.h"
#include "ddf_pool.h"
#include "ddf_device.h"
#include "ddf_fft.h"

using namespace ddf;

namespace ddf {
void set_last_error(const std::string& msg);  // ddfgpu.hip: the message ddf_last_error() returns
}

namespace {

int ifail(int code, const std::string& m) {
  ddf::set_last_error(m);
  return code;
}

#define HIP_OK(x)                                                                               \
  do {                                                                                          \
    hipError_t e_ = (x);                                                                        \
    if (e_ != hipSuccess) return ifail(DDF_EHIP, std::string(#x) + ": " + hipGetErrorString(e_)); \
  } while (0)

// ---- centred FFTs -------------------------------------------------------------------------------
__device__ __forceinline__ int fft_wrap(int i, int n) { return i >= n ? i - n : i; }

// dst[p][y][x] = scale * src[p][(y + s) % n][(x + s) % n], a wavefront per row.
__global__ __launch_bounds__(256) void shift_planes(const float2* src, float2* dst, int n, int64_t rows, int s,
                                                    float scale) {
  const int lane = threadIdx.x & 63;
  for (int64_t r = int64_t(blockIdx.x) * 4 + (threadIdx.x >> 6); r < rows; r += int64_t(gridDim.x) * 4) {
    const int y = int(r % n);
    const DDF_GLOBAL float2* in = gptr(src) + (r - y + fft_wrap(y + s, n)) * n;
    DDF_GLOBAL float2* out = gptr_w(dst) + r * n;
    for (int x0 = lane; x0 < n; x0 += 256) {
      float2 v[4];
#pragma unroll
      for (int k = 0; k < 4; ++k)
        if (x0 + 64 * k < n) v[k] = ld2(in + fft_wrap(x0 + 64 * k + s, n));
#pragma unroll
      for (int k = 0; k < 4; ++k)
        if (x0 + 64 * k < n) st2(out + x0 + 64 * k, make_float2(v[k].x * scale, v[k].y * scale));
    }
  }
}

int shift(const float2* src, float2* dst, int n, int64_t nplanes, int s, float scale, hipStream_t st) {
  const int64_t rows = nplanes * n;
  hipLaunchKernelGGL(shift_planes, dim3(unsigned(std::min<int64_t>((rows + 3) / 4, 1 << 20))), dim3(256), 0, st, src, dst, n,
                     rows, s, scale);
  HIP_OK(hipGetLastError());
  return DDF_OK;
}

// A cached rocFFT plan is read-only once made, so calls on several streams or host threads may
// share it; each call brings its own execution info, work buffer and staging buffer.
struct FFTPlan {
  rocfft_plan plan = nullptr;
  size_t work_size = 0;
};

std::mutex g_fft_mu;
std::map<std::tuple<int, int64_t, int, int>, FFTPlan> g_fft_plans;  // (n, nplanes, dir, device)

int get_plan(int n, int64_t nplanes, int inverse, FFTPlan** out) {
  int dev = 0;
  HIP_OK(hipGetDevice(&dev));
  std::lock_guard<std::mutex> lk(g_fft_mu);
  static bool setup = false;
  if (!setup) {
    if (rocfft_setup() != rocfft_status_success) return ifail(DDF_EHIP, "rocfft_setup failed");
    setup = true;
  }
  auto key = std::make_tuple(n, nplanes, inverse, dev);
  auto it = g_fft_plans.find(key);
  if (it != g_fft_plans.end()) {
    *out = &it->second;
    return DDF_OK;
  }
  FFTPlan P;
  size_t lengths[2] = {size_t(n), size_t(n)};
  if (rocfft_plan_create(&P.plan, rocfft_placement_inplace,
                         inverse ? rocfft_transform_type_complex_inverse : rocfft_transform_type_complex_forward,
                         rocfft_precision_single, 2, lengths, size_t(nplanes), nullptr) != rocfft_status_success)
    return ifail(DDF_EHIP, "rocfft_plan_create failed");
  if (rocfft_plan_get_work_buffer_size(P.plan, &P.work_size) != rocfft_status_success) {
    (void)rocfft_plan_destroy(P.plan);
    return ifail(DDF_EHIP, "rocfft work size query failed");
  }
  auto res = g_fft_plans.emplace(key, P);
  *out = &res.first->second;
  return DDF_OK;
}

// LDS of a pass: `count` transforms of n points, the twiddles and the places of the frequencies.
constexpr size_t fft_lds_bytes(int n, int count) { return size_t(n) * (count + 1) * 8 + size_t(n) * 2; }
constexpr size_t kFftLds = 80 * 1024;  // for two workgroups a CU

// Factors and device tables of a length (made once per length and device, 12 n bytes); false where the
// passes do not take it: a prime factor above 13, or a length whose strip of four columns no longer
// leaves room for two workgroups on a CU (above 1950; a strip of two is read in 16-byte pieces).  24 planes,
// passes and rocFFT: 1944 points 1.47 ms, 1.71; with one workgroup a CU 1960 points 1.98, 1.86 and 2048 points
// 2.20, 1.85.
std::map<std::pair<int, int>, FftDims> g_fft_dims;  // (n, device)

int fft_dims(int n, FftDims* out, bool* ok) {
  *ok = false;
  FftDims d{};
  d.n = n;
  int left = n, L = n;
  for (int r : {13, 11, 7, 5, 3, 8, 4, 2}) {
    while (left % r == 0 && left > 1) {
      if (d.nst == kFftStages) return DDF_OK;
      left /= r;
      L /= r;
      const int s = d.nst++;
      d.radix[s] = r;
      d.m[s] = L;
      d.rcp_m[s] = L > 1 ? uint32_t(((uint64_t(1) << 32) + L - 1) / L) : 0;
      const int nb = n / r;
      d.rcp_b[s] = nb > 1 ? uint32_t(((uint64_t(1) << 32) + nb - 1) / nb) : 0;
    }
  }
  if (left != 1 || fft_lds_bytes(n, 4) > kFftLds) return DDF_OK;
  d.rcp_n = n > 1 ? uint32_t(((uint64_t(1) << 32) + n - 1) / n) : 0;
  int dev = 0;
  HIP_OK(hipGetDevice(&dev));
  std::lock_guard<std::mutex> lk(g_fft_mu);
  auto key = std::make_pair(n, dev);
  auto it = g_fft_dims.find(key);
  if (it == g_fft_dims.end()) {
    std::vector<char> h(size_t(n) * 12);
    float2* tw = reinterpret_cast<float2*>(h.data());
    uint16_t* perm = reinterpret_cast<uint16_t*>(h.data() + size_t(n) * 8);
    for (int k = 0; k < n; ++k) {
      const double a = -2. * 3.14159265358979323846 * double(k) / double(n);
      tw[k] = make_float2(float(std::cos(a)), float(std::sin(a)));
      int p = 0, r = k;
      for (int s = 0; s < d.nst; ++s) {
        p += (r % d.radix[s]) * d.m[s];
        r /= d.radix[s];
      }
      perm[k] = uint16_t(p);
    }
    void* t = nullptr;
    HIP_OK(hipMalloc(&t, h.size()));
    if (hipMemcpy(t, h.data(), h.size(), hipMemcpyHostToDevice) != hipSuccess) {
      (void)hipFree(t);
      return ifail(DDF_EHIP, "uploading the FFT tables failed");
    }
    d.tw = static_cast<const float2*>(t);
    d.perm = reinterpret_cast<const uint16_t*>(static_cast<char*>(t) + size_t(n) * 8);
    it = g_fft_dims.emplace(key, d).first;
  }
  *out = it->second;
  *ok = true;
  return DDF_OK;
}

// ---- facet geometry (GiveEdges, DDFacet/ToolsDir/GiveEdges.py:29-82, Parity=None) -------------
struct Edges {
  int x0m, x1m, y0m, y1m, x0f, x1f, y0f, y1f;
};

Edges give_edges(int xc, int yc, int m, int nfacet) {
  Edges e;
  const int h = nfacet / 2;
  int mx0 = xc - h;
  e.x0m = mx0 > 0 ? mx0 : 0;
  e.x0f = e.x0m - mx0;
  int mx1 = xc + h;
  int x1m = mx1 < m - 1 ? mx1 : m - 1;
  e.x1f = nfacet - (mx1 - x1m);
  e.x1m = x1m + 1;
  int my0 = yc - h;
  e.y0m = my0 > 0 ? my0 : 0;
  e.y0f = e.y0m - my0;
  int my1 = yc + h;
  int y1m = my1 < m - 1 ? my1 : m - 1;
  e.y1f = nfacet - (my1 - y1m);
  e.y1m = y1m + 1;
  return e;
}

struct ImgFacet {
  Edges e;
  const float* sphe;
  const float* inv_sphe;
  const float* sw;
  const float2* dirty;
  float2* model;
  const double* sumwt;
  const double* sum_jones;
};

// FacetNorm[X, Y] = sum over facets (in order) of SW_f[a, b]
__global__ __launch_bounds__(256) void facet_norm_kernel(const ImgFacet* F, int nf, int n, int m, float* norm) {
  for (int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x; i < int64_t(m) * m;
       i += int64_t(gridDim.x) * blockDim.x) {
    const int X = int(i / m), Y = int(i - int64_t(X) * m);
    float acc = 0.f;
    for (int f = 0; f < nf; ++f) {
      const Edges& e = F[f].e;
      if (X < e.x0m || X >= e.x1m || Y < e.y0m || Y >= e.y1m) continue;
      const int a = X - e.x0m + e.x0f, b = Y - e.y0m + e.y0f;
      if (a < e.x0f || a >= e.x1f || b < e.y0f || b >= e.y1f) continue;
      acc = acc + F[f].sw[size_t(a) * n + b];
    }
    norm[i] = acc;
  }
}

// Sums over the facets that cover a main-image pixel, in facet order.
//   kStitch   Image[ch, pol, X, Y] = sum_f Im_f / FacetNorm, with Im_f[a, b] = Im[n-1-b, a] (the
//             Im[::-1, :].T of the reference) and Im[i, j] = Re(dirty) * InvSphe * SW_grid / weights in
//             FP64, stored FP32, zero where Sphe < 1e-3.  SW_grid[n-1-b, a] = SW[a, b].
//   kCutAdj   adjoint of the model cut: image_bar[ch, pol, X, Y] = sum_f factor / FacetNorm[X, Y] *
//             SW[a, b] / Sphe[a, b] * Re(plane_bar[ch, pol, n-1-b, a]), zero where Sphe < 1e-3 (the
//             forward's flips and box read backwards).  The plane comes before the last shift of its
//             transform and its scale: element (i, j) is at ((i + shift) % n, (j + shift) % n), times
//             `scale`.
// Bound: HBM, the real parts of the covering facets' planes (whole lines of complex values) and one
// pass over their tapers.  A facet plane runs along X and the image along Y, so a workgroup takes 32 x
// 32 pixels and turns each facet's tile over in LDS: both sides are read along their rows.  It first
// lists the facets whose box meets its tile (a pixel has 3-4 of them, whatever their number) and takes
// up to PL planes of one facet at a time, which share the taper, its inverse and SW.  121 facets of
// 975^2, 4 bands: 1.8 ms (2.4 in tiles of 32 x 32); 16.3 with a lane per pixel testing every facet.
enum GatherMode { kStitch, kCutAdj };
template <GatherMode MODE, int PL, int T>
__global__ __launch_bounds__(256) void facet_gather(const ImgFacet* F, int nf, int n, int nband, int npol, int m,
                                                    const float* norm, const int* use_norm, float factor, int shift,
                                                    float scale, float* image) {
  constexpr int R = T * T / 256, DY = 256 / T;  // pixels of a thread, DY rows apart
  using V = typename std::conditional<MODE == kStitch, double, float>::type;
  __shared__ V tile[PL][T][T + 1];
  __shared__ uint8_t keep[T][T + 1];
  __shared__ double s_w[PL];
  __shared__ int s_list[256];
  __shared__ int s_cnt[4];
  const int t = threadIdx.x, tx = t % T, ty = t / T;
  const int tiles = (m + T - 1) / T;
  const int X0 = int(blockIdx.x % unsigned(tiles)) * T, Y0 = blockIdx.y * T;
  const int nplane = nband * npol, plane0 = int(blockIdx.x / unsigned(tiles)) * PL, np = min(PL, nplane - plane0);
  const size_t nn = size_t(n) * n;
  float acc[PL][R];
#pragma unroll
  for (int p = 0; p < PL; ++p)
#pragma unroll
    for (int i = 0; i < R; ++i) acc[p][i] = 0.f;
  for (int f0 = 0; f0 < nf; f0 += 256) {
    // the facets of this batch that meet the tile, in order
    bool hit = false;
    if (f0 + t < nf) {
      const Edges e = F[f0 + t].e;
      hit = X0 < e.x1m && X0 + T > e.x0m && Y0 < e.y1m && Y0 + T > e.y0m;
    }
    const uint64_t mask = __ballot(hit);
    if ((t & 63) == 0) s_cnt[t >> 6] = __popcll(mask);
    __syncthreads();
    int before = 0, count = 0;
    for (int w = 0; w < 4; ++w) {
      if (w < (t >> 6)) before += s_cnt[w];
      count += s_cnt[w];
    }
    if (hit) s_list[before + __popcll(mask & ((1ull << (t & 63)) - 1))] = f0 + t;
    __syncthreads();
    for (int k = 0; k < count; ++k) {
      const ImgFacet fa = F[s_list[k]];
      const Edges& e = fa.e;
      // along the facet's rows: lanes are X
#pragma unroll
      for (int i = 0; i < R; ++i) {
        const int X = X0 + tx, yl = ty + DY * i, Y = Y0 + yl;
        if (X < e.x0m || X >= e.x1m || Y < e.y0m || Y >= e.y1m) continue;
        const int a = X - e.x0m + e.x0f, b = Y - e.y0m + e.y0f;
        const size_t g = size_t(n - 1 - b) * n + a;
        if (MODE == kStitch) {
          keep[yl][tx] = !(fa.sphe[g] < 1e-3f);
          const double inv = double(fa.inv_sphe[g]);
#pragma unroll
          for (int p = 0; p < PL; ++p)
            if (p < np) tile[p][yl][tx] = V(double(fa.dirty[(plane0 + p) * nn + g].x) * inv);
        } else {
#pragma unroll
          for (int p = 0; p < PL; ++p)
            if (p < np) tile[p][yl][tx] = fa.model[(plane0 + p) * nn + size_t(fft_wrap(n - 1 - b + shift, n)) * n + fft_wrap(a + shift, n)].x * scale;
        }
      }
      if (MODE == kStitch && t < np) {
        const int plane = plane0 + t, ch = plane / npol;
        double w = fa.sumwt[plane];
        double sjn = 1.0;
        if (fa.sum_jones) {
          double ssq = fa.sum_jones[nband + ch];
          if (ssq == 0.) ssq = 1.;
          sjn = fa.sum_jones[ch] / ssq;
          if (sjn == 0.) sjn = 1.;
        }
        w = w * sqrt(sjn);
        s_w[t] = w == 0. ? 1.0 : w;
      }
      __syncthreads();
      // along the image's rows: lanes are Y
#pragma unroll
      for (int i = 0; i < R; ++i) {
        const int xl = ty + DY * i, X = X0 + xl, Y = Y0 + tx;
        if (X < e.x0m || X >= e.x1m || Y < e.y0m || Y >= e.y1m) continue;
        const int a = X - e.x0m + e.x0f, b = Y - e.y0m + e.y0f;
        const size_t ab = size_t(a) * n + b;
        if (MODE == kStitch) {
          if (!keep[tx][xl]) continue;
          const double sw = double(fa.sw[ab]);
#pragma unroll
          for (int p = 0; p < PL; ++p)
            if (p < np) acc[p][i] = acc[p][i] + float(double(tile[p][tx][xl]) * sw / s_w[p]);
        } else {
          const float sp = fa.sphe[ab];
          if (sp < 1e-3f) continue;
          const float sw = fa.sw[ab], nm = norm[size_t(X) * m + Y];
#pragma unroll
          for (int p = 0; p < PL; ++p)
            if (p < np) acc[p][i] = acc[p][i] + float(tile[p][tx][xl]) * factor / nm * sw / sp;
        }
      }
      __syncthreads();
    }
  }
  const bool divide = MODE == kStitch && *use_norm;
#pragma unroll
  for (int i = 0; i < R; ++i) {
    const int X = X0 + ty + DY * i, Y = Y0 + tx;
    if (X >= m || Y >= m) continue;
    const size_t pix = size_t(X) * m + Y;
    const float nm = divide ? norm[pix] : 1.f;
#pragma unroll
    for (int p = 0; p < PL; ++p)
      if (p < np) image[size_t(plane0 + p) * m * m + pix] = divide ? acc[p][i] / nm : acc[p][i];
  }
}

// Model grid (before the FFT) of a facet: B[i, j] = A[j, n-1-i] (A.T[::-1, :]) with
// A[a, b] = Image[ch, pol, x0d + a - x0p, y0d + b - y0p] / FacetNorm * SW[a, b] / Sphe[a, b]
// inside the facet box, 0 outside and where Sphe < 1e-3, then * (OverS * n)^2.  A plane whose
// cut is entirely zero is left zero without normalisation (ClassImToGrid.py:175-176).
struct CutP {
  const float* image;
  const float* norm;
  const int* plane_nz;  // [facet][plane]
  int m, nplane;
  float factor;
};

// The cut of every facet into its planes, as the forward transform takes it: element (y, x) of a plane
// is the model grid's element ((y + s) % n, (x + s) % n).  The image, its norm and the facet's weights
// run along the grid's columns, so a workgroup turns 32 x 32 elements over in LDS, four planes of the
// facet at a time, which share norm, SW and Sphe.  Bound: HBM (one write of the planes).  121 facets of
// 975^2 in 4 bands: 9.9 ms with a lane per element reading the image across its rows, 2.2 here.
constexpr int kCutTile = 32;
__global__ __launch_bounds__(256) void model_cut_kernel(const ImgFacet* F, int n, int shift, CutP c) {
  constexpr int T = kCutTile, R = T / 8, PL = 4;
  __shared__ float tile[PL][T][T + 1];
  const int tiles = (n + T - 1) / T;
  const int f = int(blockIdx.x / unsigned(tiles));
  const int x0 = int(blockIdx.x - unsigned(f) * unsigned(tiles)) * T, y0 = blockIdx.y * T;
  const int tx = threadIdx.x % T, ty = threadIdx.x / T;
  const ImgFacet fa = F[f];
  const Edges& e = fa.e;
  DDF_GLOBAL float2* o = gptr_w(fa.model);
  // this thread's elements of the image: pixel (-1: outside the facet's box or zero by its taper),
  // norm, SW and Sphe
  int64_t pix[R];
  float nm[R], sw[R], sp[R];
#pragma unroll
  for (int i = 0; i < R; ++i) {
    const int y = y0 + tx, x = x0 + ty + 8 * i;
    pix[i] = -1;
    nm[i] = sw[i] = sp[i] = 1.f;
    if (y >= n || x >= n) continue;
    const int a = fft_wrap(x + shift, n), b = n - 1 - fft_wrap(y + shift, n);
    if (a < e.x0f || a >= e.x1f || b < e.y0f || b >= e.y1f) continue;
    const size_t ab = size_t(a) * n + b;
    sp[i] = gptr(fa.sphe)[ab];
    sw[i] = gptr(fa.sw)[ab];
    const int64_t at = int64_t(e.x0m + a - e.x0f) * c.m + (e.y0m + b - e.y0f);
    nm[i] = gptr(c.norm)[at];
    if (!(sp[i] < 1e-3f)) pix[i] = at;
  }
  for (int p0 = 0; p0 < c.nplane; p0 += PL) {
#pragma unroll
    for (int p = 0; p < PL; ++p) {
      const bool nz = p0 + p < c.nplane && c.plane_nz[f * c.nplane + p0 + p] != 0;
#pragma unroll
      for (int i = 0; i < R; ++i) {
        float v = 0.f;
        if (nz && pix[i] >= 0) {
          v = gptr(c.image)[int64_t(p0 + p) * c.m * c.m + pix[i]];
          v = v / nm[i];
          v = v * sw[i];
          v = v / sp[i];
          v = v * c.factor;
        }
        tile[p][ty + 8 * i][tx] = v;
      }
    }
    __syncthreads();
#pragma unroll
    for (int p = 0; p < PL; ++p) {
      if (p0 + p >= c.nplane) break;
#pragma unroll
      for (int i = 0; i < R; ++i) {
        const int y = y0 + ty + 8 * i, x = x0 + tx;
        if (y < n && x < n) st2(o + (size_t(p0 + p) * n + y) * n + x, make_float2(tile[p][tx][ty + 8 * i], 0.f));
      }
    }
    __syncthreads();
  }
}

// plane_nz[facet][plane]: whether the facet's box of the plane has a value other than zero.  A
// workgroup stops once the flag is up, so a plane with sources is read only in part.
__global__ __launch_bounds__(256) void model_nonzero_kernel(const ImgFacet* F, int nplane, int m, const float* image,
                                                            int split, int* plane_nz) {
  const unsigned k = blockIdx.x / unsigned(split);  // `split` workgroups per (facet, plane)
  const Edges e = F[k / unsigned(nplane)].e;
  const int plane = int(k % unsigned(nplane)), w = e.x1m - e.x0m, h = e.y1m - e.y0m;
  int* flag = plane_nz + k;
  for (int x = int(blockIdx.x - k * unsigned(split)); x < w; x += split) {
    if (__hip_atomic_load(flag, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) return;
    const float* row = image + (size_t(plane) * m + e.x0m + x) * m + e.y0m;
    bool nz = false;
    for (int y = threadIdx.x; y < h; y += blockDim.x) nz |= row[y] != 0.f;
    if (__ballot(nz)) {
      if ((threadIdx.x & 63) == 0) __hip_atomic_store(flag, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      return;
    }
  }
}

// ---- the passes of the centred FFTs ---------------------------------------------------------------
// A 2-D transform is a pass over columns and one over rows, each reading and writing the plane once,
// in place: the shifts of the centred transform are index offsets of a pass's loads and stores and the
// scale is applied by the last store.  Bound: HBM; a strip of C columns holds n C values in LDS, C such
// that two workgroups share a CU, and is read in C * 8-byte pieces.  Loads are issued eight at a time
// before their LDS stores.  484 planes of 975^2 (3.7 GB each way): columns 3.0 ms, rows 2.5 ms; the
// rocFFT plan with its transposes and the shifts around it 9.1 together.
struct FftPass {
  int shift_in, shift_out;  // element j takes source (j + shift_in) % n; result p is frequency (p + shift_out) % n
  int inverse;
  float scale;
};
constexpr int kFftBatch = 8;

// LDS of a pass: the values, the twiddles and the places of the frequencies.
struct FftLds {
  float2 *buf, *tw;
  uint16_t* perm;
};
__device__ __forceinline__ FftLds fft_lds_setup(float2* lds, const FftDims& d, int count) {
  FftLds l{lds, lds + d.n * count, reinterpret_cast<uint16_t*>(lds + d.n * (count + 1))};
  for (int i = threadIdx.x; i < d.n; i += blockDim.x) {
    l.tw[i] = d.tw[i];
    l.perm[i] = d.perm[i];
  }
  return l;
}

template <int LOGC>
__global__ __launch_bounds__(512) void fft_columns(FftDims d, float2* planes, FftPass fp, int strips) {
  extern __shared__ __attribute__((aligned(16))) float2 fft_lds[];
  constexpr int C = 1 << LOGC, T = 512;
  const int n = d.n;
  const int64_t plane = blockIdx.x / strips;
  const int x0 = int(blockIdx.x - plane * strips) * C;
  DDF_GLOBAL float2* data = gptr_w(planes + size_t(plane) * n * n) + x0;
  const int c = threadIdx.x & (C - 1);  // T is a multiple of C: a lane keeps its column
  const bool in = x0 + c < n;
  const FftLds l = fft_lds_setup(fft_lds, d, C);
  for (int i0 = threadIdx.x; i0 < n * C; i0 += kFftBatch * T) {
    float2 v[kFftBatch];
#pragma unroll
    for (int k = 0; k < kFftBatch; ++k) {
      const int i = i0 + k * T;
      v[k] = make_float2(0.f, 0.f);
      if (in && i < n * C) v[k] = ld2(data + size_t(fft_wrap((i >> LOGC) + fp.shift_in, n)) * n + c);
    }
#pragma unroll
    for (int k = 0; k < kFftBatch; ++k)
      if (i0 + k * T < n * C) l.buf[i0 + k * T] = make_float2(v[k].x, fp.inverse ? -v[k].y : v[k].y);
  }
  __syncthreads();
  fft_stages<true>(l.buf, l.tw, d, C, LOGC, 1, C);
  if (!in) return;
  const float si = fp.inverse ? -fp.scale : fp.scale;
  for (int i0 = threadIdx.x; i0 < n * C; i0 += kFftBatch * T) {
#pragma unroll
    for (int k = 0; k < kFftBatch; ++k) {
      const int i = i0 + k * T;
      if (i < n * C) {
        const float2 v = l.buf[(int(l.perm[fft_wrap((i >> LOGC) + fp.shift_out, n)]) << LOGC) + c];
        st2(data + size_t(i >> LOGC) * n + c, make_float2(v.x * fp.scale, v.y * si));
      }
    }
  }
}

// `rows` rows of the planes per workgroup (rows of all planes follow one another).
__global__ __launch_bounds__(256) void fft_rows(FftDims d, float2* planes, FftPass fp, int rows, int64_t total) {
  extern __shared__ __attribute__((aligned(16))) float2 fft_lds[];
  constexpr int T = 256;
  const int n = d.n;
  const int64_t r0 = int64_t(blockIdx.x) * rows;
  const int count = int(total - r0 < rows ? total - r0 : rows), all = count * n;
  DDF_GLOBAL float2* data = gptr_w(planes + size_t(r0) * n);
  const FftLds l = fft_lds_setup(fft_lds, d, rows);
  for (int i0 = threadIdx.x; i0 < all; i0 += kFftBatch * T) {
    float2 v[kFftBatch];
#pragma unroll
    for (int k = 0; k < kFftBatch; ++k) {
      const int i = i0 + k * T;
      v[k] = make_float2(0.f, 0.f);
      if (i < all) {
        const int at = __mul24(fft_div(i, n, d.rcp_n), n);
        v[k] = ld2(data + at + fft_wrap(i - at + fp.shift_in, n));
      }
    }
#pragma unroll
    for (int k = 0; k < kFftBatch; ++k)
      if (i0 + k * T < all) l.buf[i0 + k * T] = make_float2(v[k].x, fp.inverse ? -v[k].y : v[k].y);
  }
  __syncthreads();
  fft_stages<false>(l.buf, l.tw, d, count, 0, n, 1);
  const float si = fp.inverse ? -fp.scale : fp.scale;
  for (int i0 = threadIdx.x; i0 < all; i0 += kFftBatch * T) {
#pragma unroll
    for (int k = 0; k < kFftBatch; ++k) {
      const int i = i0 + k * T;
      if (i < all) {
        const int at = __mul24(fft_div(i, n, d.rcp_n), n);
        const float2 v = l.buf[at + int(l.perm[fft_wrap(i - at + fp.shift_out, n)])];
        st2(data + i, make_float2(v.x * fp.scale, v.y * si));
      }
    }
  }
}

// flag: whether any of x is other than zero.  A wavefront looks at the flag first, stores it once and
// stops where it is up (a store a lane, all to one word, took 9.4 ms for a 6237^2 image).
__global__ __launch_bounds__(256) void any_nonzero_kernel(const float* x, int64_t n, int* flag) {
  for (int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x; i < n; i += int64_t(gridDim.x) * blockDim.x) {
    if (__hip_atomic_load(flag, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) return;
    const uint64_t nz = __ballot(x[i] != 0.f);
    if (!nz) continue;
    if ((threadIdx.x & 63) == __builtin_ctzll(nz)) __hip_atomic_store(flag, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    return;
  }
}

__global__ void zero_ints(int* x, int n) {
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) x[i] = 0;
}

unsigned blocks_for(int64_t n) {
  int64_t b = (n + 255) / 256;
  if (b > 65536) b = 65536;
  if (b < 1) b = 1;
  return unsigned(b);
}

// planes: where the model planes are, `per` values a facet, in place of the facets' own (null: those)
int upload_facets(const ddf_image_facet* facets, int nf, int n, int m, hipStream_t st, ImgFacet** dout,
                  std::vector<void*>& tmp, float2* planes = nullptr, int64_t per = 0) {
  std::vector<ImgFacet> h(static_cast<size_t>(nf));
  for (int i = 0; i < nf; ++i) {
    const ddf_image_facet& f = facets[i];
    if (!f.sphe || !f.sw) return ifail(DDF_EINVAL, "facet Sphe / SW pointer is null");
    h[size_t(i)].e = give_edges(f.xc, f.yc, m, n);
    h[size_t(i)].sphe = f.sphe;
    h[size_t(i)].inv_sphe = f.inv_sphe;
    h[size_t(i)].sw = f.sw;
    h[size_t(i)].dirty = reinterpret_cast<const float2*>(f.dirty);
    h[size_t(i)].model = planes ? planes + i * per : reinterpret_cast<float2*>(f.model);
    h[size_t(i)].sumwt = f.sumwt;
    h[size_t(i)].sum_jones = f.sum_jones;
    const Edges& e = h[size_t(i)].e;
    if (e.x1m <= e.x0m || e.y1m <= e.y0m || e.x0f < 0 || e.y0f < 0 || e.x1f > n || e.y1f > n ||
        e.x1f - e.x0f != e.x1m - e.x0m || e.y1f - e.y0f != e.y1m - e.y0m)
      return ifail(DDF_EINVAL, "facet box does not intersect the main image consistently");
  }
  void* d = nullptr;
  HIP_OK(ddf::pool_alloc(&d, h.size() * sizeof(ImgFacet), st));
  tmp.push_back(d);
  HIP_OK(hipMemcpyAsync(d, h.data(), h.size() * sizeof(ImgFacet), hipMemcpyHostToDevice, st));
  *dout = static_cast<ImgFacet*>(d);
  return DDF_OK;
}

// The centred transform of `nplanes` planes by the passes.  Columns of a strip: the most of 16, 8 and 4
// that leave two workgroups a CU (80 KB of LDS each: 16 to 593 points, 8 to 1107, 4 to 1950); rows of a
// workgroup: about 32 KB, at most 16.  Fewer rows where the launch would not give every CU two workgroups: a
// transform of one plane of 189^2 17-21 us, 26 with 16 rows; 36 of 525^2 123, 156 with a row (a line at 128 to 2048
// workgroups is equal).
int fft_planes(const FftDims& d, float2* planes, int64_t nplanes, int inverse, double scale, hipStream_t st) {
  const int n = d.n;
  const double norm = inverse ? scale : scale / (double(n) * double(n));
  FftPass fp{n / 2, (n + 1) / 2, inverse != 0, 1.f};
  int lc = 4;
  while (fft_lds_bytes(n, 1 << lc) > kFftLds) --lc;  // (fft_dims: a strip of four fits)
  const int strips = (n + (1 << lc) - 1) >> lc;
  int rows = int(32 * 1024 / (size_t(n) * 8));
  rows = int(std::max<int64_t>(1, std::min<int64_t>({16, rows, nplanes * n / 512})));
  const dim3 b(512);
  const size_t lds = fft_lds_bytes(n, 1 << lc);
  // a launch takes fewer than 2^32 threads: 2^22 strips of 512 at most, and no more rows than fit as well
  const int64_t most = (int64_t(1) << 22) / strips;
  for (int64_t p0 = 0; p0 < nplanes; p0 += most) {
    const int64_t np = std::min(most, nplanes - p0), nrow = np * n;
    float2* a = planes + p0 * n * n;
    const dim3 g(unsigned(np * strips));
    fp.scale = 1.f;
    if (lc == 4) hipLaunchKernelGGL((fft_columns<4>), g, b, lds, st, d, a, fp, strips);
    else if (lc == 3) hipLaunchKernelGGL((fft_columns<3>), g, b, lds, st, d, a, fp, strips);
    else hipLaunchKernelGGL((fft_columns<2>), g, b, lds, st, d, a, fp, strips);
    HIP_OK(hipGetLastError());
    fp.scale = float(norm);
    hipLaunchKernelGGL(fft_rows, dim3(unsigned((nrow + rows - 1) / rows)), dim3(256), fft_lds_bytes(n, rows), st, d, a, fp,
                       rows, nrow);
    HIP_OK(hipGetLastError());
  }
  return DDF_OK;
}

template <GatherMode MODE>
int launch_gather(const ImgFacet* F, int nf, int n, int nband, int npol, int m, const float* norm, const int* use_norm,
                  float factor, int shift, float scale, float* image, hipStream_t st) {
  // A plane alone: 16 x 16 pixels up to 1536 tiles of 32 x 32, which read longer pieces of the facets.  Stitch of
  // 945^2 from 9 facets 93 us with 16, 98 with 32; 1575^2 of 25 223, 219; 3645^2 of 81 690, 654.  Planes together:
  // 16 x 16, whose LDS lets more workgroups onto a CU: 243^2, 9 facets x 4 planes 88 us, 124 with 32; 6237^2, 121
  // x 4 2.53 ms, 3.10.
  const unsigned groups = (unsigned(nband) * unsigned(npol) + 3) / 4, t32 = unsigned((m + 31) / 32), t16 = unsigned((m + 15) / 16);
  const bool one = nband * npol == 1, large = one && uint64_t(t32) * t32 > 1536;
  const unsigned tiles = large ? t32 : t16;
  const dim3 g(tiles * groups, tiles), b(256);
  if (large)
    hipLaunchKernelGGL((facet_gather<MODE, 1, 32>), g, b, 0, st, F, nf, n, nband, npol, m, norm, use_norm, factor, shift,
                       scale, image);
  else if (one)
    hipLaunchKernelGGL((facet_gather<MODE, 1, 16>), g, b, 0, st, F, nf, n, nband, npol, m, norm, use_norm, factor, shift,
                       scale, image);
  else
    hipLaunchKernelGGL((facet_gather<MODE, 4, 16>), g, b, 0, st, F, nf, n, nband, npol, m, norm, use_norm, factor, shift,
                       scale, image);
  HIP_OK(hipGetLastError());
  return DDF_OK;
}

struct TmpFree {
  std::vector<void*>& v;
  hipStream_t st;
  ~TmpFree() {
    for (void* p : v) (void)hipFreeAsync(p, st);
  }
};

}  // namespace

// Per-call resources of the rocFFT transforms, released on every return path (stream-ordered frees).
struct FFTCall {
  hipStream_t st;
  void* tmp = nullptr;
  void* work = nullptr;
  rocfft_execution_info info = nullptr;
  ~FFTCall() {
    if (info) (void)rocfft_execution_info_destroy(info);
    if (work) (void)hipFreeAsync(work, st);
    if (tmp) (void)hipFreeAsync(tmp, st);
  }
  // tmp of `total` values and what the plan wants
  int setup(FFTPlan* P, int64_t total) {
    HIP_OK(ddf::pool_alloc(&tmp, size_t(total) * sizeof(float2), st));
    if (rocfft_execution_info_create(&info) != rocfft_status_success)
      return ifail(DDF_EHIP, "rocfft_execution_info_create failed");
    if (P->work_size) {
      HIP_OK(ddf::pool_alloc(&work, P->work_size, st));
      if (rocfft_execution_info_set_work_buffer(info, work, P->work_size) != rocfft_status_success)
        return ifail(DDF_EHIP, "rocfft work buffer failed");
    }
    if (rocfft_execution_info_set_stream(info, st) != rocfft_status_success) return ifail(DDF_EHIP, "rocfft stream");
    return DDF_OK;
  }
  int run(FFTPlan* P, void* data) {
    void* bufs[1] = {data};
    if (rocfft_execute(P->plan, bufs, nullptr, info) != rocfft_status_success) return ifail(DDF_EHIP, "rocfft_execute failed");
    return DDF_OK;
  }
};

// The transforms of the facet models and of their adjoint keep the 2-D rocFFT plans, one over the planes of
// every facet where those follow one another in memory and one a facet elsewhere: their rounding is in the
// predicted visibilities, and an FP64 loss that a program forms of those moves by some 1e-8 with another
// transform (two 1-D plans with transposes between them round differently at 33 to 135, 243 and 343 points of
// the odd lengths from 33 to 2025, though not at the others).
struct ModelPlanes {
  int groups;       // calls of the transform
  int64_t nplanes;  // planes of one
  FFTPlan* plan = nullptr;
  bool joined() const { return groups == 1; }
  float2* at(const ddf_image_facet* facets, int k) const { return reinterpret_cast<float2*>(facets[k].model); }
  ModelPlanes(const ddf_image_facet* facets, int nf, int n, int64_t per) {
    bool contiguous = true;
    for (int f = 1; f < nf; ++f) contiguous &= at(facets, f) == at(facets, 0) + f * per * n * n;
    groups = contiguous ? 1 : nf;
    nplanes = (nf / groups) * per;
  }
  int setup(FFTCall* call, int n, int inverse) {
    int rc = get_plan(n, nplanes, inverse, &plan);
    return rc ? rc : call->setup(plan, nplanes * n * n);
  }
};

extern "C" int ddf_fft2c(float* planes, int32_t n, int64_t nplanes, int32_t inverse, double scale, void* stream) {
  if (!planes || n <= 0 || nplanes <= 0) return ifail(DDF_EINVAL, "bad FFT arguments");
  hipStream_t st = static_cast<hipStream_t>(stream);
  FftDims dims;
  bool own = false;
  int rc = fft_dims(n, &dims, &own);
  if (rc) return rc;
  if (own) return fft_planes(dims, reinterpret_cast<float2*>(planes), nplanes, inverse, scale, st);
  FFTPlan* P = nullptr;
  rc = get_plan(n, nplanes, inverse, &P);
  if (rc) return rc;
  const int64_t total = int64_t(n) * n * nplanes;
  FFTCall call{st};
  if ((rc = call.setup(P, total))) return rc;
  float2* a = reinterpret_cast<float2*>(planes);
  float2* t = static_cast<float2*>(call.tmp);
  // ifftshift: t[j] = a[(j + n/2) % n]
  if ((rc = shift(a, t, n, nplanes, n / 2, 1.f, st)) || (rc = call.run(P, t))) return rc;
  // fftshift: a[k] = t[(k + (n+1)/2) % n], with the normalisation
  double norm = inverse ? scale : scale / (double(n) * double(n));
  return shift(t, a, n, nplanes, (n + 1) / 2, float(norm), st);
}

extern "C" int ddf_facet_norm(const ddf_image_facet* facets, int32_t nf, int32_t npix_facet, int32_t m,
                              float* facet_norm, void* stream) {
  if (!facets || nf <= 0 || npix_facet <= 0 || m <= 0 || !facet_norm) return ifail(DDF_EINVAL, "bad arguments");
  hipStream_t st = static_cast<hipStream_t>(stream);
  std::vector<void*> tmp;
  TmpFree guard{tmp, st};
  ImgFacet* d = nullptr;
  int rc = upload_facets(facets, nf, npix_facet, m, st, &d, tmp);
  if (rc) return rc;
  hipLaunchKernelGGL(facet_norm_kernel, dim3(blocks_for(int64_t(m) * m)), dim3(256), 0, st, d, nf, npix_facet, m,
                     facet_norm);
  HIP_OK(hipGetLastError());
  return DDF_OK;
}

extern "C" int ddf_stitch(const ddf_image_facet* facets, int32_t nf, int32_t npix_facet, int32_t nband, int32_t npol,
                          int32_t m, const float* facet_norm, float* image, void* stream) {
  if (!facets || nf <= 0 || npix_facet <= 0 || m <= 0 || !facet_norm || !image || nband <= 0 || npol <= 0)
    return ifail(DDF_EINVAL, "bad arguments");
  for (int i = 0; i < nf; ++i)
    if (!facets[i].dirty || !facets[i].inv_sphe || !facets[i].sumwt) return ifail(DDF_EINVAL, "facet buffer is null");
  hipStream_t st = static_cast<hipStream_t>(stream);
  // a graph would keep the address of this call's list of facets, and read it at every replay
  hipStreamCaptureStatus capture = hipStreamCaptureStatusNone;
  if (hipStreamIsCapturing(st, &capture) != hipSuccess) (void)hipGetLastError();
  if (capture != hipStreamCaptureStatusNone) return ifail(DDF_EHIP, "ddf_stitch cannot be captured into a graph");
  std::vector<void*> tmp;
  TmpFree guard{tmp, st};
  ImgFacet* d = nullptr;
  int rc = upload_facets(facets, nf, npix_facet, m, st, &d, tmp);
  if (rc) return rc;
  // "if (FacetNorm != 0).any(): Image /= FacetNorm"
  int* flag = nullptr;
  HIP_OK(ddf::pool_alloc(reinterpret_cast<void**>(&flag), sizeof(int), st));
  tmp.push_back(flag);
  hipLaunchKernelGGL(zero_ints, dim3(1), dim3(64), 0, st, flag, 1);
  hipLaunchKernelGGL(any_nonzero_kernel, dim3(unsigned(std::min<int64_t>(256, 1 + int64_t(m) * m / 16384))), dim3(256), 0, st, facet_norm,
                     int64_t(m) * m, flag);
  HIP_OK(hipGetLastError());
  return launch_gather<kStitch>(d, nf, npix_facet, nband, npol, m, facet_norm, flag, 0.f, 0, 1.f, image, st);
}

extern "C" int ddf_model_to_grid(const ddf_image_facet* facets, int32_t nf, int32_t npix_facet, int32_t nband,
                                 int32_t npol, int32_t m, const float* image, const float* facet_norm, int32_t overs,
                                 void* stream) {
  if (!facets || nf <= 0 || npix_facet <= 0 || m <= 0 || !image || !facet_norm || nband <= 0 || npol <= 0)
    return ifail(DDF_EINVAL, "bad arguments");
  for (int i = 0; i < nf; ++i)
    if (!facets[i].model) return ifail(DDF_EINVAL, "facet model pointer is null");
  hipStream_t st = static_cast<hipStream_t>(stream);
  const int n = npix_facet, per = nband * npol;
  ModelPlanes mp(facets, nf, n, per);
  FFTCall call{st};
  int rc = mp.setup(&call, n, 0);
  if (rc) return rc;
  float2* t = static_cast<float2*>(call.tmp);
  std::vector<void*> tmp;
  TmpFree guard{tmp, st};
  ImgFacet* d = nullptr;
  // the cut goes straight to where the transform takes it
  rc = upload_facets(facets, nf, n, m, st, &d, tmp, mp.joined() ? t : nullptr, int64_t(per) * n * n);
  if (rc) return rc;
  int* nz = nullptr;
  HIP_OK(ddf::pool_alloc(reinterpret_cast<void**>(&nz), sizeof(int) * size_t(per) * nf, st));
  tmp.push_back(nz);
  const float factor = float(double(overs) * n) * float(double(overs) * n);
  const CutP cut{image, facet_norm, nz, m, per, factor};
  hipLaunchKernelGGL(zero_ints, dim3(blocks_for(int64_t(per) * nf)), dim3(256), 0, st, nz, per * nf);
  // workgroups of a plane: one per 16384 values (a store to the flag for each, where the plane has sources)
  const int split = int(std::min<int64_t>(64, 1 + int64_t(n) * n / 16384));
  hipLaunchKernelGGL(model_nonzero_kernel, dim3(unsigned(per) * unsigned(nf) * unsigned(split)), dim3(256), 0, st, d, per, m,
                     image, split, nz);
  HIP_OK(hipGetLastError());
  const unsigned cuts = unsigned((n + kCutTile - 1) / kCutTile);
  hipLaunchKernelGGL(model_cut_kernel, dim3(unsigned(nf) * cuts, cuts), dim3(256), 0, st, d, n, n / 2, cut);
  HIP_OK(hipGetLastError());
  for (int k = 0; k < mp.groups; ++k) {
    float2* a = mp.at(facets, k);
    if (!mp.joined() && (rc = shift(a, t, n, mp.nplanes, 0, 1.f, st))) return rc;
    if ((rc = call.run(mp.plan, t)) ||
        (rc = shift(t, a, n, mp.nplanes, (n + 1) / 2, float(1.0 / (double(n) * double(n))), st)))
      return rc;
  }
  return DDF_OK;
}

extern "C" int ddf_model_to_grid_adjoint(const ddf_image_facet* facets, int32_t nf, int32_t npix_facet, int32_t nband,
                                         int32_t npol, int32_t m, float* image_bar, const float* facet_norm,
                                         int32_t overs, void* stream) {
  if (!facets || nf <= 0 || npix_facet <= 0 || m <= 0 || !image_bar || !facet_norm || nband <= 0 || npol <= 0)
    return ifail(DDF_EINVAL, "bad arguments");
  for (int i = 0; i < nf; ++i)
    if (!facets[i].model) return ifail(DDF_EINVAL, "facet model pointer is null");
  hipStream_t st = static_cast<hipStream_t>(stream);
  const int n = npix_facet;
  // adjoint of the forward centred FFT (1/n^2 fft): the centred inverse FFT scaled by 1/n^2; where the planes
  // follow one another the gather takes the last shift and the scale
  const int64_t per = int64_t(nband) * npol;
  const float scale = float(1.0 / (double(n) * double(n)));
  ModelPlanes mp(facets, nf, n, per);
  FFTCall call{st};
  int rc = mp.setup(&call, n, 1);
  if (rc) return rc;
  float2* t = static_cast<float2*>(call.tmp);
  for (int k = 0; k < mp.groups; ++k) {
    float2* a = mp.at(facets, k);
    if ((rc = shift(a, t, n, mp.nplanes, n / 2, 1.f, st)) || (rc = call.run(mp.plan, t))) return rc;
    if (!mp.joined() && (rc = shift(t, a, n, mp.nplanes, (n + 1) / 2, scale, st))) return rc;
  }
  std::vector<void*> tmp;
  TmpFree guard{tmp, st};
  ImgFacet* d = nullptr;
  rc = upload_facets(facets, nf, n, m, st, &d, tmp, mp.joined() ? t : nullptr, per * n * n);
  if (rc) return rc;
  const float factor = float(double(overs) * n) * float(double(overs) * n);
  return launch_gather<kCutAdj>(d, nf, n, nband, npol, m, facet_norm, nullptr, factor, mp.joined() ? (n + 1) / 2 : 0,
                                mp.joined() ? scale : 1.f, image_bar, st);
}
