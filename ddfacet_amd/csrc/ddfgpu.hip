// gfx950 facet gridder / degridder: plain single-facet kernels and the C ABI of include/ddfgpu.h.
//
// Work decomposition (one facet per launch, the "plain" path):
//   * a wavefront takes 1, 8 or 64 BDA blocks, by the map's mean visibilities per block (grid-stride);
//   * a block's (row, channel) visibilities are spread over its lanes, channel fastest;
//   * block sums (visibility, uvw means, weights) are reduced across a block's lanes by butterfly
//     shuffles; the w-plane / cell / oversampling decision is then uniform over them;
//   * gridding scatters the S x S x npol stamps, a whole wavefront per stamp, through global float
//     atomics; degridding gathers the same stamp, reduces it, and writes every (row, channel)
//     of the block back once (blocks of a degrid map are disjoint).
//   * sumwt / SumJones / SumJonesChan go through per-workgroup LDS accumulators flushed once per
//     workgroup with global FP64 atomics.
// Follows gridder::gridder (DDFacet/Gridder/gridder.h:78-377) and degridder::degridder
// (degridder.h:55-266); argument dispatch follows GridderSmearPols.cc:76-348.
#include <hip/hip_runtime.h>

#include <cstdio>
#include <cstring>
#include <mutex>
#include <string>
#include <algorithm>
#include <cmath>
#include <vector>

#include "../../include/ddfgpu.h"
#include "ddf_device.h"
#include "ddf_internal.h"

using namespace ddf;

namespace {

thread_local std::string g_err;

int fail(int code, const std::string& msg) {
  g_err = msg;
  return code;
}

#define HIP_TRY(expr)                                                                \
  do {                                                                               \
    hipError_t e_ = (expr);                                                          \
    if (e_ != hipSuccess) return fail(DDF_EHIP, std::string(#expr) + ": " + hipGetErrorString(e_)); \
  } while (0)

// ---- correlation <-> Stokes maps (Stokes.h), as 4x4 complex matrices -----------------------
struct StokesMap {
  int read;        // 4, 2, 1: Read_4Corr / Read_2Corr_Pad / Read_1Corr_Pad
  int nstokes;
  double m[4][4][2];
};

bool same(const uint16_t* c, int n, std::initializer_list<int> w) {
  if (n != int(w.size())) return false;
  int i = 0;
  for (int x : w)
    if (c[i++] != x) return false;
  return true;
}

std::string stokes_string(const ddf_vis* v) {
  std::string s;
  for (int i = 0; i < v->nstokes; ++i) s += (v->stokes_codes[i] >= 1 && v->stokes_codes[i] <= 4) ? "?IQUV"[v->stokes_codes[i]] : '!';
  return s;
}

void set(double (&m)[4][4][2], int r, int c, double re, double im) {
  m[r][c][0] = re;
  m[r][c][1] = im;
}

// Grid side, GridderSmearPols.cc:128-206 with the Stokes.h:18-34 formulas.
int grid_map(const ddf_vis* v, StokesMap* sm) {
  const uint16_t* c = v->corr_codes;
  int nc = v->ncorr_codes;
  for (int i = 0; i < nc; ++i)
    if (!((c[i] >= 5 && c[i] <= 12) || c[i] == 1))
      return fail(DDF_EINVAL, "Only accepts I,RR,RL,LR,LL,XX,XY,YX,YY as correlation input type");
  for (int i = 0; i < v->nstokes; ++i)
    if (v->stokes_codes[i] < 1 || v->stokes_codes[i] > 4)
      return fail(DDF_EINVAL, "Only accepts I,Q,U,V as polarization output type");
  std::memset(sm, 0, sizeof(*sm));
  std::string want = stokes_string(v), eff = want;
  int kind;  // 0 circular 4-corr, 1 linear 4-corr, 2 linear 2-corr, 3 circular 2-corr, 4 Stokes I
  std::vector<std::string> ok;
  if (same(c, nc, {9, 10, 11, 12})) { kind = 1; sm->read = 4; ok = {"I", "Q", "U", "V", "IQ", "IU", "IV", "QU", "IQU", "IQUV"}; }
  else if (same(c, nc, {5, 6, 7, 8})) { kind = 0; sm->read = 4; ok = {"I", "IQ", "IU", "IV", "QU", "IQU", "IQUV"}; }
  else if (same(c, nc, {9, 12})) { kind = 2; sm->read = 2; ok = {"I", "IQ"}; }
  else if (same(c, nc, {5, 8})) { kind = 3; sm->read = 2; ok = {"I", "IV"}; }
  else if (same(c, nc, {1})) { kind = 4; sm->read = 1; ok = {"I"}; }
  else return fail(DDF_EINVAL, "Cannot convert input correlations to desired output Stokes parameters.");
  bool found = false;
  for (auto& o : ok) found |= (o == want);
  if (!found) return fail(DDF_EINVAL, "Cannot convert input correlations to desired output Stokes parameters.");
  if (kind == 1 && want == "IU") eff = "IQ";  // the {I,U} request runs the IQ policy (GridderSmearPols.cc:142-143)
  sm->nstokes = v->nstokes;
  for (int k = 0; k < sm->nstokes; ++k) {
    char s = eff[k];
    auto& m = sm->m;
    if (kind == 4) { set(m, k, 0, 1, 0); continue; }
    if (s == 'I') { set(m, k, 0, .5, 0); set(m, k, 3, .5, 0); continue; }
    bool lin = (kind == 1 || kind == 2);
    if ((lin && s == 'Q') || (!lin && s == 'V')) { set(m, k, 0, .5, 0); set(m, k, 3, -.5, 0); }
    else if ((lin && s == 'U') || (!lin && s == 'Q')) { set(m, k, 1, .5, 0); set(m, k, 2, .5, 0); }
    else { set(m, k, 1, 0, -.5); set(m, k, 2, 0, .5); }  // V (linear) / U (circular): -(c1-c2)*0.5i
  }
  return DDF_OK;
}

// Degrid side, GridderSmearPols.cc:261-342 with the Stokes.h:90-192 formulas.
int degrid_map(const ddf_vis* v, StokesMap* sm) {
  const uint16_t* c = v->corr_codes;
  int nc = v->ncorr_codes;
  for (int i = 0; i < nc; ++i)
    if (!((c[i] >= 5 && c[i] <= 12) || c[i] == 1))
      return fail(DDF_EINVAL, "Only accepts I,RR,RL,LR,LL,XX,XY,YX,YY as correlation output types");
  std::memset(sm, 0, sizeof(*sm));
  std::string w = stokes_string(v);
  bool X4 = same(c, nc, {9, 10, 11, 12}), R4 = same(c, nc, {5, 6, 7, 8});
  bool X2 = same(c, nc, {9, 12}), R2 = same(c, nc, {5, 8}), S1 = same(c, nc, {1});
  auto& m = sm->m;
  // rows: correlation slot (2x2 flattened), columns: Stokes index
  if (w == "I" && (X4 || X2 || R4 || R2 || S1)) { set(m, 0, 0, 1, 0); set(m, 3, 0, 1, 0); }
  else if (w == "Q" && X4) { set(m, 0, 0, 1, 0); set(m, 3, 0, -1, 0); }
  else if (w == "U" && X4) { set(m, 1, 0, 1, 0); set(m, 2, 0, 1, 0); }
  else if (w == "V" && X4) { set(m, 1, 0, 0, 1); set(m, 2, 0, 0, -1); }
  else if (w == "IQUV" && X4) { set(m, 0, 0, 1, 0); set(m, 0, 1, 1, 0); set(m, 1, 2, 1, 0); set(m, 1, 3, 0, 1);
                                set(m, 2, 2, 1, 0); set(m, 2, 3, 0, -1); set(m, 3, 0, 1, 0); set(m, 3, 1, -1, 0); }
  else if (w == "IQUV" && R4) { set(m, 0, 0, 1, 0); set(m, 0, 3, 1, 0); set(m, 1, 1, 1, 0); set(m, 1, 2, 0, 1);
                                set(m, 2, 1, 1, 0); set(m, 2, 2, 0, -1); set(m, 3, 0, 1, 0); set(m, 3, 3, -1, 0); }
  else if (w == "IQ" && (X4 || X2)) { set(m, 0, 0, 1, 0); set(m, 0, 1, 1, 0); set(m, 3, 0, 1, 0); set(m, 3, 1, -1, 0); }
  else if (w == "IQ" && R4) { set(m, 0, 0, 1, 0); set(m, 1, 1, 1, 0); set(m, 2, 1, 1, 0); set(m, 3, 0, 1, 0); }
  else if (w == "IU" && X4) { set(m, 0, 0, 1, 0); set(m, 1, 1, 1, 0); set(m, 2, 1, 1, 0); set(m, 3, 0, 1, 0); }
  else if (w == "IU" && R4) { set(m, 0, 0, 1, 0); set(m, 1, 1, 0, 1); set(m, 2, 1, 0, -1); set(m, 3, 0, 1, 0); }
  else if (w == "IV" && (R4 || R2)) { set(m, 0, 0, 1, 0); set(m, 0, 1, 1, 0); set(m, 3, 0, 1, 0); set(m, 3, 1, -1, 0); }
  else if (w == "IV" && X4) { set(m, 0, 0, 1, 0); set(m, 1, 1, 0, 1); set(m, 2, 1, 0, -1); set(m, 3, 0, 1, 0); }
  else if (w == "QU" && X4) { set(m, 0, 0, 1, 0); set(m, 1, 1, 1, 0); set(m, 2, 1, 1, 0); set(m, 3, 0, -1, 0); }
  else if (w == "IQU" && X4) { set(m, 0, 0, 1, 0); set(m, 0, 1, 1, 0); set(m, 1, 2, 1, 0); set(m, 2, 2, 1, 0);
                               set(m, 3, 0, 1, 0); set(m, 3, 1, -1, 0); }
  else if (w == "IQU" && R4) { set(m, 0, 0, 1, 0); set(m, 1, 1, 1, 0); set(m, 1, 2, 0, 1); set(m, 2, 1, 1, 0);
                               set(m, 2, 2, 0, -1); set(m, 3, 0, 1, 0); }
  else return fail(DDF_EINVAL, "Cannot convert input Stokes parameter to desired output correlations.");
  sm->read = (X4 || R4) ? 4 : ((X2 || R2) ? 2 : 1);
  sm->nstokes = v->nstokes;
  return DDF_OK;
}

// ---- kernel parameters -----------------------------------------------------------------------
struct KParams {
  VisP v;
  void* grid;
  int nband, npol, ny, nx;
  double incr0, incr1;
  int dopsf;
  double cu, cv, l0, m0, n0;
  double fmean0, wl_mean;
  double tscale0;  // decorr_tscale(fmean0)
  CFP cf;
  JonesP jp;
  DecorrP dp;
  double* sumwt;
  int nstokes;
  double sm[4][4][2];
  int chan_lds;   // per-channel Jones sums accumulated in LDS (else straight to global)
  int64_t large;       // visibilities of a large block: the first large_wgs workgroups take those
  unsigned large_wgs;
};

__device__ __forceinline__ cd smc(const KParams& p, int r, int c) { return cd{p.sm[r][c][0], p.sm[r][c][1]}; }

// ---- the plain kernels ---------------------------------------------------------------------
// A wavefront takes 64 / GS consecutive blocks, GS = 1 << LG lanes each: the lanes of a group walk their
// block's rows and visibilities (channel fastest) and add up their partial sums by a butterfly within
// the group; then the whole wavefront takes the stamps of its blocks one after the other, lanes over
// cells, the next stamp's CF values in flight with the current one.  GS follows the map's mean visibilities
// per block (plain_group): with a wavefront per block, a block of one visibility left 63 lanes idle through
// the phase, the Jones products and the placement.  An averaging map has blocks of hundreds of visibilities
// beside its single ones: with 1 or 8 lanes a block these are left to the first workgroups of the launch,
// which look through the map and give each a wavefront.
template <int LG>
__device__ __forceinline__ double group_sum(double v) {
#pragma unroll
  for (int o = 1; o < (1 << LG); o <<= 1) v += __shfl_xor(v, o, kWave);
  return v;
}
template <int LG>
__device__ __forceinline__ int group_sum(int v) {
#pragma unroll
  for (int o = 1; o < (1 << LG); o <<= 1) v += __shfl_xor(v, o, kWave);
  return v;
}
__device__ __forceinline__ int read_lane(int x, int j) { return __builtin_amdgcn_readlane(x, j); }
__device__ __forceinline__ int64_t read_lane(int64_t x, int j) {
  return int64_t(uint64_t(uint32_t(read_lane(int(uint32_t(uint64_t(x))), j))) |
                 (uint64_t(uint32_t(read_lane(int(uint32_t(uint64_t(x) >> 32)), j))) << 32));
}
__device__ __forceinline__ double read_lane(double x, int j) {
  return __builtin_bit_cast(double, read_lane(__builtin_bit_cast(int64_t, x), j));
}

// The wavefronts of a part of the launch, and this one's place among them.
struct Part {
  int64_t wave, nwaves;
};
template <int LG>
__device__ __forceinline__ Part plain_part(const KParams& p, bool large) {
  const unsigned wgs = LG == 6 ? gridDim.x : large ? p.large_wgs : gridDim.x - p.large_wgs;
  const unsigned wg = LG == 6 || large ? blockIdx.x : blockIdx.x - p.large_wgs;
  return Part{(int64_t(wg) * blockDim.x + threadIdx.x) >> 6, (int64_t(wgs) * blockDim.x) >> 6};
}
// The kernel's parameters, read again: with one set of loads for both parts of a launch the compiler holds them over the
// branch and spills for it.
__device__ __forceinline__ const KParams& own_params() {
  auto q = __builtin_amdgcn_kernarg_segment_ptr();
  asm volatile("" : "+s"(q));
  return *(const KParams*)q;
}
// The large ones of the blocks b0, b0 + nwaves, ... (neighbours, often of one baseline and large together, go to
// different wavefronts so).
__device__ __forceinline__ uint64_t large_blocks(const KParams& p, int64_t b0, int64_t nwaves) {
  const int64_t b = b0 + (threadIdx.x & 63) * nwaves;
  const BlockRec br = read_block(p.v, b < p.v.nblocks ? b : 0);
  return __ballot(b < p.v.nblocks && int64_t(br.nr) * (br.ch1 - br.ch0) > p.large);
}

// Block means over the unflagged (row, channel) visibilities (gridder.h:272-289).
struct Means {
  double su, sv, sw, sf;
  int cnt;
};
template <int LG>
__device__ inline Means block_means(const KParams& p, const BlockRec& br, int64_t nvis, int sub) {
  const VisP& v = p.v;
  const int nch = br.ch1 - br.ch0;
  Means m{0, 0, 0, 0, 0};
  for (int64_t k = sub; k < nvis; k += 1 << LG) {
    const int r = int(k / nch);
    const int c = br.ch0 + int(k - int64_t(r) * nch);
    const int64_t row = br.rows[r];
    if (row < 0 || row >= v.nrow) continue;
    if (gptr(v.flags)[(size_t(row) * v.nchan + c) * v.ncorr]) continue;
    const DDF_GLOBAL double* uvw = gptr(v.uvw) + 3 * row;
    m.su += shifted(uvw[0], uvw[2], p.cu);
    m.sv += shifted(uvw[1], uvw[2], p.cv);
    m.sw += uvw[2];
    m.sf += gptr(v.freqs)[c];
    ++m.cnt;
  }
  m.cnt = group_sum<LG>(m.cnt);
  m.su = group_sum<LG>(m.su);
  m.sv = group_sum<LG>(m.sv);
  m.sw = group_sum<LG>(m.sw);
  m.sf = group_sum<LG>(m.sf);
  return m;
}

// ---- gridding kernel -----------------------------------------------------------------------
// The scatter is bound by the atomics' cache lines: neighbouring lanes take the real and imaginary part
// of one cell, so that a line of the grid is touched once a stamp and not once for either part.
// 561 600 blocks of one visibility, 7 x 7 stamps: 1.60 ms with a wavefront per block, 0.51 here
// (0.19 of it without the atomics; 0.64 with 8 lanes per block).
template <int READ, int JMODE, typename GT, int LG, bool LARGE>
__device__ __forceinline__ void grid_part(const KParams& p, const Part& part, double* s_sumwt, double* s_sj, double* s_sjc) {
  constexpr int GS = 1 << LG, NB = kWave / GS;
  const int lane = threadIdx.x & 63, sub = lane & (GS - 1), grp = lane >> LG;
  const int64_t wave = part.wave, nwaves = part.nwaves;
  const VisP& v = p.v;
  DDF_GLOBAL GT* grid = gptr_w(reinterpret_cast<GT*>(p.grid));
  const int npg = p.nstokes < p.npol ? p.nstokes : p.npol;
  double* sjc = p.chan_lds ? s_sjc : p.jp.sum_jones_chan;

  auto block = [&](int64_t b) {  // of this group of lanes
    const bool mine = b < v.nblocks && !(v.sparse && !v.sparse[b]);
    const BlockRec br = read_block(v, mine ? b : 0);
    const int nch = br.ch1 - br.ch0;
    const int64_t size = int64_t(br.nr) * nch;
    const int64_t nvis = mine && (LG == 6 || size <= p.large) ? size : 0;
    const int64_t mid = nvis > 0 ? int64_t(br.rows[br.nr / 2]) : -1;
    const bool mid_ok = mid >= 0 && mid < v.nrow;
    const double dec = mid_ok ? decorr_factor(p.dp, v.uvw, p.tscale0, mid) : 1.;
    const int gchan = nvis > 0 ? gptr(v.chan_map)[br.ch0] : -1;

    // With Jones the per-channel sums are only added for gridded blocks, so the placement is
    // decided first from a means-only pass (the same partial sums the main pass forms).
    Place pl{0, 0, 0, 0, 0};
    bool decided = false;
    double BBblk = 0;
    JonesPair jblk;
    if (JMODE != 0) {
      const Means m = block_means<LG>(p, br, nvis, sub);
      const double um = m.su / m.cnt, vm = m.sv / m.cnt, wm = m.sw / m.cnt, fm = m.sf / m.cnt;
      decided = m.cnt > 0 && gchan >= 0 && gchan < p.nband &&
                place_block(p.cf, p.nx, p.ny, p.incr0, p.incr1, um, vm, wm, fm / kC, &pl);
      if (JMODE == 2 && decided) {
        double uvwm[3] = {um, vm, wm};
        jblk = jones_at(p.jp, mid_ok ? mid : 0, (br.ch0 + br.ch1) / 2, uvwm, p.wl_mean);
        BBblk = jblk.BB;
      }
    }

    double su = 0, sv = 0, sw = 0, sf = 0, swt = 0, ssw = 0, sj = 0;
    int cnt = 0;
    cd acc[4] = {{0, 0}, {0, 0}, {0, 0}, {0, 0}};
    for (int64_t k = sub; k < (JMODE == 0 || decided ? nvis : 0); k += GS) {
      const int r = int(k / nch);
      const int c = br.ch0 + int(k - int64_t(r) * nch);
      const int64_t row = br.rows[r];
      if (row < 0 || row >= v.nrow) continue;
      const size_t vc = size_t(row) * v.nchan + c;
      if (gptr(v.flags)[vc * v.ncorr]) continue;
      const double* uvw = v.uvw + 3 * row;
      const double U = gptr(uvw)[0], V = gptr(uvw)[1], W = gptr(uvw)[2];
      const double f = gptr(v.freqs)[c];
      const double fw = double(gptr(v.weights)[vc]);
      const double fwd = fw * dec * dec;
      cd meas[4];
      if (p.dopsf) {
        meas[0] = cd{dec, 0}; meas[1] = cd{0, 0}; meas[2] = cd{0, 0}; meas[3] = cd{dec, 0};
      } else {
        const DDF_GLOBAL float2* vp = gptr(v.vis) + vc * v.ncorr;
        if (READ == 4) {
#pragma unroll
          for (int q = 0; q < 4; ++q) meas[q] = cd{vp[q].x, vp[q].y};
        } else if (READ == 2) {
          meas[0] = cd{vp[0].x, vp[0].y}; meas[1] = cd{0, 0}; meas[2] = cd{0, 0}; meas[3] = cd{vp[1].x, vp[1].y};
        } else {
          meas[0] = cd{vp[0].x, vp[0].y}; meas[1] = cd{0, 0}; meas[2] = cd{0, 0}; meas[3] = meas[0];
        }
      }
      cd wt = cd{fw, 0};
      if (!p.dopsf) {
        const double angle = -2. * kPi * (U * p.l0 + V * p.m0 + W * p.n0) / kC;
        wt = phasor(f * angle) * fw;
      }
      if (JMODE == 1) {
        JonesPair jj = jones_at(p.jp, row, c, uvw, p.wl_mean);
        M2 m;
        if (p.dopsf) {
          m = mul(mul(herm(jj.J0), mul(jj.J0, herm(jj.J1))), jj.J1);
#pragma unroll
          for (int q = 0; q < 4; ++q) m.a[q] = m.a[q] * dec;
        } else {
          m = mul(mul(herm(jj.J0), M2{{meas[0], meas[1], meas[2], meas[3]}}), jj.J1);
        }
#pragma unroll
        for (int q = 0; q < 4; ++q) meas[q] = m.a[q];
        sj += jj.BB * fwd;
        atomicAdd(&sjc[c], double(npg) * (jj.BB * fwd));
      }
      if (JMODE == 2) atomicAdd(&sjc[c], double(npg) * (fwd * BBblk));
      if (JMODE != 0) atomicAdd(&sjc[v.nchan + c], double(npg) * fwd);
      if (READ == 4) {
#pragma unroll
        for (int q = 0; q < 4; ++q) acc[q] = acc[q] + meas[q] * wt;
      } else if (READ == 2) {
        acc[0] = acc[0] + meas[0] * wt;
        acc[3] = acc[3] + meas[3] * wt;
      } else {
        acc[0] = acc[0] + meas[0] * wt;
      }
      if (JMODE == 0) {
        su += shifted(U, W, p.cu);
        sv += shifted(V, W, p.cv);
        sw += W;
        sf += f;
        ++cnt;
      }
      swt += fw;
      ssw += fwd;
    }
    if (JMODE == 0) {
      cnt = group_sum<LG>(cnt);
      su = group_sum<LG>(su); sv = group_sum<LG>(sv); sw = group_sum<LG>(sw); sf = group_sum<LG>(sf);
      decided = cnt > 0 && gchan >= 0 && gchan < p.nband &&
                place_block(p.cf, p.nx, p.ny, p.incr0, p.incr1, su / cnt, sv / cnt, sw / cnt, (sf / cnt) / kC, &pl);
    }
    swt = group_sum<LG>(swt);
    ssw = group_sum<LG>(ssw);
    if (JMODE == 1) sj = group_sum<LG>(sj);
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      if (READ == 4 || q == 0 || (READ == 2 && q == 3)) {
        acc[q].re = group_sum<LG>(acc[q].re);
        acc[q].im = group_sum<LG>(acc[q].im);
      }
    }
    if (JMODE == 2 && decided) {
      M2 m{{acc[0], acc[1], acc[2], acc[3]}};
      if (p.dopsf) m = mul(mul(jblk.J0, m), herm(jblk.J1));
      m = mul(mul(herm(jblk.J0), m), jblk.J1);
#pragma unroll
      for (int q = 0; q < 4; ++q) acc[q] = m.a[q];
      sj = ssw * BBblk;
    }
    if (decided && sub == 0) {
      for (int ip = 0; ip < npg; ++ip) {
        atomicAdd(&s_sumwt[gchan * p.npol + ip], swt);
        if (JMODE != 0) {
          atomicAdd(&s_sj[gchan], sj);
          atomicAdd(&s_sj[gchan + p.nband], ssw);
        }
      }
    }
    // the stamps: element t of a stamp is part t & 1 of cell t >> 1
    const int64_t first = ((int64_t(gchan) * p.npol) * p.ny + (pl.locy - pl.sup)) * p.nx + (pl.locx - pl.sup);
    uint64_t todo = __ballot(decided && sub == 0);
    auto cf_of = [&](int j, float2 (&w)[2]) {
      const int S = read_lane(pl.S, j), n2 = 2 * S * S;
      const DDF_GLOBAL float2* cf = gptr(p.cf.data) + read_lane(pl.cfoff, j);
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        w[h] = make_float2(0.f, 0.f);
        if (lane + 64 * h < n2) w[h] = ld2(cf + ((lane + 64 * h) >> 1));
      }
    };
    float2 wn[2] = {make_float2(0.f, 0.f), make_float2(0.f, 0.f)};
    if (todo) cf_of(__builtin_ctzll(todo), wn);
    while (todo) {
      const int j = __builtin_ctzll(todo);
      todo &= todo - 1;
      const float2 w0 = wn[0], w1 = wn[1];
      if (todo) cf_of(__builtin_ctzll(todo), wn);
      const int S = read_lane(pl.S, j), n2 = 2 * S * S;
      const int64_t base = read_lane(first, j);
      const DDF_GLOBAL float2* cf = gptr(p.cf.data) + read_lane(pl.cfoff, j);
      const float invS = __builtin_amdgcn_rcpf(float(S));
      cd a[4];
#pragma unroll
      for (int q = 0; q < 4; ++q) a[q] = cd{read_lane(acc[q].re, j), read_lane(acc[q].im, j)};
      for (int ip = 0; ip < npg; ++ip) {
        cd st = cd{0, 0};
#pragma unroll
        for (int q = 0; q < 4; ++q) st = st + smc(p, ip, q) * a[q];
        // part 0: re w.x - im w.y, part 1: re w.y + im w.x
        const double si = (lane & 1) ? st.im : -st.im;
        DDF_GLOBAL GT* g = grid + 2 * (base + int64_t(ip) * p.ny * p.nx) + (lane & 1);
        for (int t = lane; t < n2; t += kWave) {
          const float2 w = t < 64 ? w0 : (t < 128 ? w1 : ld2(cf + (t >> 1)));
          const int k = t >> 1;
          // (k + 0.5) / S is at least 0.5 / S from an integer: exact for S < 32
          const int sy = S < 32 ? int((float(k) + 0.5f) * invS) : k / S, sx = k - sy * S;
          const double x = st.re * double((lane & 1) ? w.y : w.x) + si * double((lane & 1) ? w.x : w.y);
          atomic_add_g(g + 2 * (int64_t(sy) * p.nx + sx), GT(x));
        }
      }
    }
  };
  for (int64_t b0 = wave * NB; b0 < v.nblocks; b0 += nwaves * (LARGE ? kWave : NB)) {
    if (LARGE) {
      for (uint64_t take = large_blocks(p, b0, nwaves); take; take &= take - 1) block(b0 + __builtin_ctzll(take) * nwaves);
    } else {
      block(b0 + grp);
    }
  }
}

template <int READ, int JMODE, typename GT, int LG>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2))) void grid_plain(KParams p) {
  extern __shared__ double lds[];
  const int nbp = p.nband * p.npol;
  double* s_sumwt = lds;                       // [nband*npol]
  double* s_sj = lds + nbp;                    // [2*nband]
  double* s_sjc = lds + nbp + 2 * p.nband;     // [2*nchan] when chan_lds
  const int nacc = nbp + 2 * p.nband + (p.chan_lds ? 2 * p.v.nchan : 0);
  for (int i = threadIdx.x; i < nacc; i += blockDim.x) lds[i] = 0.;
  __syncthreads();
  if (LG < 6 && blockIdx.x < p.large_wgs) {
    const KParams& q = own_params();
    grid_part<READ, JMODE, GT, 6, true>(q, plain_part<LG>(q, true), s_sumwt, s_sj, s_sjc);
  } else
    grid_part<READ, JMODE, GT, LG, false>(p, plain_part<LG>(p, false), s_sumwt, s_sj, s_sjc);
  __syncthreads();
  for (int i = threadIdx.x; i < nbp; i += blockDim.x)
    if (s_sumwt[i] != 0.) atomicAdd(&p.sumwt[i], s_sumwt[i]);
  if (JMODE != 0) {
    for (int i = threadIdx.x; i < 2 * p.nband; i += blockDim.x)
      if (s_sj[i] != 0.) atomicAdd(&p.jp.sum_jones[i], s_sj[i]);
    if (p.chan_lds)
      for (int i = threadIdx.x; i < 2 * p.v.nchan; i += blockDim.x)
        if (s_sjc[i] != 0.) atomicAdd(&p.jp.sum_jones_chan[i], s_sjc[i]);
  }
}

// ---- degridding kernel ---------------------------------------------------------------------
// Bound by the FP64 phase and Jones products of every visibility.  Stamps of up to 256 cells are gathered with the
// next block's values in flight.  2.25 M visibilities in 509 000 blocks with DD Jones: 1.72 ms with a wavefront
// per block, 0.36 with 8 lanes and no large blocks apart, 0.27 here.
// (Three wavefronts per SIMD with Jones: the FP64 products held 253 registers, 375 us against 399 with 8 lanes.)
template <int NCORR, int JMODE, int LG, bool LARGE>
__device__ __forceinline__ void degrid_part(const KParams& p, const Part& part) {
  constexpr int GS = 1 << LG, NB = kWave / GS;
  const int lane = threadIdx.x & 63, sub = lane & (GS - 1), grp = lane >> LG;
  const int64_t wave = part.wave, nwaves = part.nwaves;
  const VisP& v = p.v;
  const DDF_GLOBAL float2* grid = gptr(reinterpret_cast<const float2*>(p.grid));

  auto block = [&](int64_t b) {  // of this group of lanes
    const BlockRec br = read_block(v, b < v.nblocks ? b : 0);
    const int nch = br.ch1 - br.ch0;
    const bool some = b < v.nblocks && br.nr > 0 && nch > 0 && (LG == 6 || int64_t(br.nr) * nch <= p.large);
    const int gchan = some ? gptr(v.chan_map)[br.ch0] : -1;
    const bool mine = some && gchan >= 0 && gchan < p.nband;
    double fm = 0;
    for (int c = br.ch0; c < (mine ? br.ch1 : br.ch0); ++c) fm += gptr(v.freqs)[c];
    fm /= double(nch);
    double su = 0, sv = 0, sw = 0;
    int cnt = 0;
    for (int r = sub; r < (mine ? br.nr : 0); r += GS) {
      const int64_t row = br.rows[r];
      if (row < 0 || row >= v.nrow) continue;
      const DDF_GLOBAL double* uvw = gptr(v.uvw) + 3 * row;
      su += shifted(uvw[0], uvw[2], p.cu);
      sv += shifted(uvw[1], uvw[2], p.cv);
      sw += uvw[2];
      ++cnt;
    }
    cnt = group_sum<LG>(cnt);
    su = group_sum<LG>(su); sv = group_sum<LG>(sv); sw = group_sum<LG>(sw);
    Place pl{0, 0, 0, 0, 0};
    const bool placed =
        cnt > 0 && place_block(p.cf, p.nx, p.ny, p.incr0, p.incr1, su / cnt, sv / cnt, sw / cnt, fm / kC, &pl);
    // gather the S x S stamp of every Stokes plane: FP32 products summed in FP64 (degridder.h:202-212)
    const int64_t first = ((int64_t(gchan) * p.npol) * p.ny + (pl.locy - pl.sup)) * p.nx + (pl.locx - pl.sup);
    cd st[4] = {{0, 0}, {0, 0}, {0, 0}, {0, 0}};
    constexpr int H = 4;
    auto load = [&](int j, int ip, float2 (&g)[H], float2 (&w)[H]) {
      const int S = read_lane(pl.S, j), S2 = S * S;
      const DDF_GLOBAL float2* cf = gptr(p.cf.data) + read_lane(pl.cfoff, j);
      const DDF_GLOBAL float2* q = grid + (read_lane(first, j) + int64_t(ip) * p.ny * p.nx);
      const float invS = __builtin_amdgcn_rcpf(float(S));
#pragma unroll
      for (int h = 0; h < H; ++h) {
        const int k = lane + 64 * h;
        g[h] = w[h] = make_float2(0.f, 0.f);
        if (k < S2) {
          const int sy = S < 32 ? int((float(k) + 0.5f) * invS) : k / S;
          g[h] = ld2(q + (int64_t(sy) * p.nx + (k - sy * S)));
          w[h] = ld2(cf + k);
        }
      }
    };
    const uint64_t all = __ballot(placed && sub == 0);
    for (int ip = 0; ip < p.nstokes; ++ip) {
      uint64_t todo = all;
      float2 gn[H], wn[H];
      if (todo) load(__builtin_ctzll(todo), ip, gn, wn);
      while (todo) {
        const int j = __builtin_ctzll(todo);
        todo &= todo - 1;
        double re = 0, im = 0;
        auto add = [&](float2 g, float2 w) {
          const float pr = g.x * w.x - g.y * w.y;
          const float pi = g.x * w.y + g.y * w.x;
          re += double(pr);
          im += double(pi);
        };
        float2 gc[H], wc[H];
#pragma unroll
        for (int h = 0; h < H; ++h) {
          gc[h] = gn[h];
          wc[h] = wn[h];
        }
        if (todo) load(__builtin_ctzll(todo), ip, gn, wn);
        const int S = read_lane(pl.S, j), S2 = S * S;
#pragma unroll
        for (int h = 0; h < H; ++h)
          if (64 * h < S2) {  // (one branch a wavefront: without it the compiler selects, and adds all H every time)
            if (lane + 64 * h < S2) add(gc[h], wc[h]);
          }
        if (S2 > 64 * H) {
          const DDF_GLOBAL float2* cf = gptr(p.cf.data) + read_lane(pl.cfoff, j);
          const DDF_GLOBAL float2* q = grid + (read_lane(first, j) + int64_t(ip) * p.ny * p.nx);
          for (int k = lane + 64 * H; k < S2; k += kWave) {
            const int sy = k / S;
            add(ld2(q + (int64_t(sy) * p.nx + (k - sy * S))), ld2(cf + k));
          }
        }
        re = wave_total(re);
        im = wave_total(im);
        if (grp == (j >> LG)) {
#pragma unroll
          for (int q = 0; q < 4; ++q)
            if (q == ip) st[q] = cd{re, im};
        }
      }
    }
    if (!placed) return;
    M2 cv;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      cv.a[k] = cd{0, 0};
#pragma unroll
      for (int q = 0; q < 4; ++q) cv.a[k] = cv.a[k] + smc(p, k, q) * st[q];
    }
    const int64_t mid = br.rows[br.nr / 2];
    const bool mid_ok = mid >= 0 && mid < v.nrow;
    if (JMODE == 2 && mid_ok) {
      JonesPair jj = jones_at(p.jp, mid, (br.ch0 + br.ch1) / 2, v.uvw + 3 * mid, p.wl_mean);
      cv = mul(mul(jj.J0, cv), herm(jj.J1));
    }
    const double dec = mid_ok ? decorr_factor(p.dp, v.uvw, decorr_tscale(fm), mid) : 1.;
    const int64_t nvis = int64_t(br.nr) * nch;
    for (int64_t k = sub; k < nvis; k += GS) {
      const int r = int(k / nch);
      const int c = br.ch0 + int(k - int64_t(r) * nch);
      const int64_t row = br.rows[r];
      if (row < 0 || row >= v.nrow) continue;
      const double* uvw = v.uvw + 3 * row;
      const double angle = 2. * kPi * (gptr(uvw)[0] * p.l0 + gptr(uvw)[1] * p.m0 + gptr(uvw)[2] * p.n0) / kC;
      const cd corr = phasor(gptr(v.freqs)[c] * angle) * dec;
      M2 vb;
      if (JMODE == 1) {
        JonesPair jj = jones_at(p.jp, row, c, uvw, p.wl_mean);
        vb = mul(mul(jj.J0, cv), herm(jj.J1));
#pragma unroll
        for (int q = 0; q < 4; ++q) vb.a[q] = vb.a[q] * corr;
      } else {
#pragma unroll
        for (int q = 0; q < 4; ++q) vb.a[q] = cv.a[q] * corr;
      }
      DDF_GLOBAL float2* vp = gptr_w(v.vis) + (size_t(row) * v.nchan + c) * NCORR;
      if (NCORR == 4) {
        float2 x[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) x[q] = ld2(vp + q);
#pragma unroll
        for (int q = 0; q < 4; ++q)
          st2(vp + q, make_float2(float(double(x[q].x) - vb.a[q].re), float(double(x[q].y) - vb.a[q].im)));
      } else if (NCORR == 2) {
        const float2 x0 = ld2(vp), x1 = ld2(vp + 1);
        st2(vp, make_float2(float(double(x0.x) - vb.a[0].re), float(double(x0.y) - vb.a[0].im)));
        st2(vp + 1, make_float2(float(double(x1.x) - vb.a[3].re), float(double(x1.y) - vb.a[3].im)));
      } else {
        const float2 x0 = ld2(vp);
        st2(vp, make_float2(float(double(x0.x) - vb.a[0].re), float(double(x0.y) - vb.a[0].im)));
      }
    }
  };
  for (int64_t b0 = wave * NB; b0 < v.nblocks; b0 += nwaves * (LARGE ? kWave : NB)) {
    if (LARGE) {
      for (uint64_t take = large_blocks(p, b0, nwaves); take; take &= take - 1) block(b0 + __builtin_ctzll(take) * nwaves);
    } else {
      block(b0 + grp);
    }
  }
}

// SPLIT: with the large blocks apart; held out where the map has none, for the registers (with Jones 119 spilled with,
// 52 without).
template <int NCORR, int JMODE, int LG, bool SPLIT>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(JMODE == 0 ? 4 : 3))) void degrid_plain(KParams p) {
  if (SPLIT && blockIdx.x < p.large_wgs) {
    const KParams& q = own_params();
    degrid_part<NCORR, JMODE, 6, true>(q, plain_part<LG>(q, true));
  } else degrid_part<NCORR, JMODE, LG, false>(p, plain_part<LG>(p, false));
}

// ---- BDA block index ---------------------------------------------------------------------------
// Word offset of every block record: start[b] = 2 + nblocks + sum_{b' < b} size[b'].
// Three phases: per-chunk sums, an exclusive scan of the chunk sums (one workgroup), and a
// per-chunk scan plus chunk offset.
constexpr int kScanChunk = 2048;

__global__ __launch_bounds__(256) void scan_chunk_sums(const int32_t* sizes, int64_t n, int64_t* chunk_sum) {
  __shared__ int64_t red[256];
  int64_t base = int64_t(blockIdx.x) * kScanChunk;
  int64_t s = 0;
  for (int i = threadIdx.x; i < kScanChunk; i += 256)
    if (base + i < n) s += sizes[base + i];
  red[threadIdx.x] = s;
  __syncthreads();
  for (int o = 128; o > 0; o >>= 1) {
    if (threadIdx.x < o) red[threadIdx.x] += red[threadIdx.x + o];
    __syncthreads();
  }
  if (threadIdx.x == 0) chunk_sum[blockIdx.x] = red[0];
}

__global__ __launch_bounds__(256) void scan_chunk_offsets(int64_t* chunk_sum, int64_t nchunk, int64_t base) {
  // exclusive scan of chunk_sum in place, one workgroup, sequential over tiles of 256
  __shared__ int64_t tile[256];
  __shared__ int64_t carry;
  if (threadIdx.x == 0) carry = base;
  __syncthreads();
  for (int64_t t0 = 0; t0 < nchunk; t0 += 256) {
    int64_t i = t0 + threadIdx.x;
    int64_t x = i < nchunk ? chunk_sum[i] : 0;
    tile[threadIdx.x] = x;
    __syncthreads();
    for (int o = 1; o < 256; o <<= 1) {
      int64_t y = threadIdx.x >= o ? tile[threadIdx.x - o] : 0;
      __syncthreads();
      tile[threadIdx.x] += y;
      __syncthreads();
    }
    if (i < nchunk) chunk_sum[i] = carry + tile[threadIdx.x] - x;
    __syncthreads();
    if (threadIdx.x == 255) carry += tile[255];
    __syncthreads();
  }
}

__global__ __launch_bounds__(256) void scan_chunk_final(const int32_t* sizes, int64_t n, const int64_t* chunk_off,
                                                        int64_t* out) {
  __shared__ int64_t tile[256];
  __shared__ int64_t carry;
  int64_t base = int64_t(blockIdx.x) * kScanChunk;
  if (threadIdx.x == 0) carry = chunk_off[blockIdx.x];
  __syncthreads();
  for (int t0 = 0; t0 < kScanChunk; t0 += 256) {
    int64_t i = base + t0 + threadIdx.x;
    int64_t x = i < n ? sizes[i] : 0;
    tile[threadIdx.x] = x;
    __syncthreads();
    for (int o = 1; o < 256; o <<= 1) {
      int64_t y = threadIdx.x >= o ? tile[threadIdx.x - o] : 0;
      __syncthreads();
      tile[threadIdx.x] += y;
      __syncthreads();
    }
    if (i < n) out[i] = carry + tile[threadIdx.x] - x;
    __syncthreads();
    if (threadIdx.x == 255) carry += tile[255];
    __syncthreads();
  }
}

// out[i] = base + sum_{j < i} x[j] (int32 in, int64 out); tmp holds ceil(n / kScanChunk) words.
int launch_scan(const int32_t* x, int64_t n, int64_t base, int64_t* out, int64_t* chunk_tmp, hipStream_t st) {
  if (n <= 0) return DDF_OK;
  int64_t nchunk = (n + kScanChunk - 1) / kScanChunk;
  hipLaunchKernelGGL(scan_chunk_sums, dim3(unsigned(nchunk)), dim3(256), 0, st, x, n, chunk_tmp);
  hipLaunchKernelGGL(scan_chunk_offsets, dim3(1), dim3(256), 0, st, chunk_tmp, nchunk, base);
  hipLaunchKernelGGL(scan_chunk_final, dim3(unsigned(nchunk)), dim3(256), 0, st, x, n, chunk_tmp, out);
  HIP_TRY(hipGetLastError());
  return DDF_OK;
}

int launch_bda_index(const int32_t* bda, int64_t nblocks, int64_t* out, int64_t* chunk_tmp, hipStream_t st) {
  return launch_scan(bda + 2, nblocks, 2 + nblocks, out, chunk_tmp, st);
}

// ---- host-side assembly ---------------------------------------------------------------------
int check_common(const ddf_grid_desc* g, const ddf_vis* v, const ddf_facet* f) {
  if (!g || !v || !f) return fail(DDF_EINVAL, "null argument struct");
  if (g->nband <= 0 || g->npol <= 0 || g->nx <= 0 || g->ny <= 0) return fail(DDF_EINVAL, "bad grid shape");
  if (!f->grid) return fail(DDF_EINVAL, "grid pointer is null");
  if (v->nrow < 0 || v->nchan <= 0 || v->ncorr <= 0 || v->ncorr > 4) return fail(DDF_EINVAL, "bad visibility shape");
  if (v->ncorr != v->ncorr_codes) return fail(DDF_EINVAL, "DataCorrFormat must list one code per correlation");
  if (v->nstokes <= 0 || v->nstokes > 4) return fail(DDF_EINVAL, "bad number of Stokes parameters");
  if (!v->uvw || !v->vis || !v->flags || !v->freqs || !v->chan_map || !v->bda)
    return fail(DDF_EINVAL, "null visibility-side pointer");
  if (v->bda_len < 2 || v->nblocks < 0 || 2 + v->nblocks > v->bda_len) return fail(DDF_EINVAL, "inconsistent BDA map");
  const ddf_cf& cf = f->cf;
  if (!cf.data || !cf.offset || !cf.support || cf.nw <= 0 || cf.overs <= 0 || cf.max_support <= 0)
    return fail(DDF_EINVAL, "bad CF table");
  if (f->jones.enabled) {
    const ddf_jones& j = f->jones;
    if (!j.kms && !j.beam)
      return fail(DDF_ERUNTIME, "Jones matricies specified but neither E or DD Jones are applied. This is a bug!");
    if (j.mode != 1 && j.mode != 2) return fail(DDF_EINVAL, "Jones mode must be 1 or 2");
    if (!j.a0 || !j.a1) return fail(DDF_EINVAL, "Jones antenna maps are null");
    if (j.kms && (!j.kms_time || !j.kms_chan)) return fail(DDF_EINVAL, "DD Jones maps are null");
    if (j.beam && (!j.beam_time || !j.beam_chan)) return fail(DDF_EINVAL, "beam Jones maps are null");
    for (int i = 0; i < 4; ++i)
      if ((j.kms && j.kms_dims[i] <= 0) || (j.beam && j.beam_dims[i] <= 0)) return fail(DDF_EINVAL, "empty Jones table");
    if (j.interp_mode == 1 && j.ncoefs > 0 && !j.coefs) return fail(DDF_EINVAL, "interpolation coefficients are null");
  }
  if (f->decorr.enabled && f->decorr.tsmear && !f->decorr.uvw_dt) return fail(DDF_EINVAL, "uvw_dt is null");
  return DDF_OK;
}

void fill_params(KParams& p, const ddf_grid_desc* g, const ddf_vis* v, const ddf_facet* f, const StokesMap& sm,
                 const int64_t* bda_start, double fmean0, double wl_mean) {
  std::memset(&p, 0, sizeof(p));
  p.v.vis = reinterpret_cast<float2*>(v->vis);
  p.v.uvw = v->uvw;
  p.v.flags = v->flags;
  p.v.weights = v->weights;
  p.v.freqs = v->freqs;
  p.v.chan_map = v->chan_map;
  p.v.nrow = v->nrow;
  p.v.nchan = v->nchan;
  p.v.ncorr = v->ncorr;
  p.v.bda = v->bda;
  p.v.bda_start = bda_start;
  p.v.nblocks = v->nblocks;
  p.v.bda_len = v->bda_len;
  p.v.sparse = v->sparsification;
  p.grid = f->grid;
  p.nband = g->nband;
  p.npol = g->npol;
  p.ny = g->ny;
  p.nx = g->nx;
  p.incr0 = g->incr[0];
  p.incr1 = g->incr[1];
  p.dopsf = g->dopsf;
  p.cu = f->cu;
  p.cv = f->cv;
  p.l0 = f->l0;
  p.m0 = f->m0;
  p.n0 = std::sqrt(1 - f->l0 * f->l0 - f->m0 * f->m0) - 1;
  p.wl_mean = wl_mean;
  p.fmean0 = fmean0;
  p.tscale0 = decorr_tscale(fmean0);
  p.cf.data = reinterpret_cast<const float2*>(f->cf.data);
  p.cf.offset = f->cf.offset;
  p.cf.support = f->cf.support;
  p.cf.nw = f->cf.nw;
  p.cf.overs = f->cf.overs;
  p.cf.ref_wave = f->cf.ref_wave;
  p.cf.wmax = f->cf.wmax;
  const ddf_jones& j = f->jones;
  p.jp.enabled = j.enabled;
  p.jp.mode = j.mode;
  p.jp.interp = j.interp_mode;
  p.jp.kms = reinterpret_cast<const float2*>(j.kms);
  p.jp.beam = reinterpret_cast<const float2*>(j.beam);
  for (int i = 0; i < 4; ++i) {
    p.jp.kdims[i] = j.kms_dims[i];
    p.jp.bdims[i] = j.beam_dims[i];
  }
  p.jp.ktime = j.kms_time;
  p.jp.kchan = j.kms_chan;
  p.jp.kdir = j.kms_dir;
  p.jp.btime = j.beam_time;
  p.jp.bchan = j.beam_chan;
  p.jp.bdir = j.beam_dir;
  p.jp.a0 = j.a0;
  p.jp.a1 = j.a1;
  p.jp.coefs = j.coefs;
  p.jp.ncoefs = j.coefs ? j.ncoefs : 0;
  p.jp.apply_amp = j.apply_amp;
  p.jp.apply_phase = j.apply_phase;
  p.jp.scale = j.scale_jones;
  p.jp.calib_error = j.calib_error;
  p.jp.sum_jones = j.sum_jones;
  p.jp.sum_jones_chan = j.sum_jones_chan;
  p.dp.enabled = f->decorr.enabled;
  p.dp.tsmear = f->decorr.tsmear;
  p.dp.fsmear = f->decorr.fsmear;
  p.dp.uvw_dt = f->decorr.uvw_dt;
  p.dp.dt = f->decorr.dt;
  p.dp.dnu = f->decorr.dnu;
  p.dp.fscale = decorr_fscale(f->decorr.dnu);
  p.dp.l0 = f->decorr.l0;
  p.dp.m0 = f->decorr.m0;
  p.sumwt = f->sumwt;
  p.nstokes = sm.nstokes;
  std::memcpy(p.sm, sm.m, sizeof(p.sm));
}

// Per-call temporary device memory (stream ordered).
struct Temp {
  hipStream_t st;
  PoolArena arena;
  explicit Temp(hipStream_t s) : st(s) {}
  void* get(size_t bytes) { return arena.get(bytes, st); }
  template <typename T>
  T* get(size_t n) { return static_cast<T*>(arena.get(n * sizeof(T), st)); }
  void free() { arena.release_all(st); }
  ~Temp() { free(); }
};

int resolve_block_index(const ddf_vis* v, Temp& tmp, const int64_t** out) {
  if (v->bda_start) {
    *out = v->bda_start;
    return DDF_OK;
  }
  if (v->nblocks == 0) {
    *out = nullptr;
    return DDF_OK;
  }
  int64_t nchunk = (v->nblocks + kScanChunk - 1) / kScanChunk;
  int64_t* starts = static_cast<int64_t*>(tmp.get(size_t(v->nblocks) * 8));
  int64_t* chunks = static_cast<int64_t*>(tmp.get(size_t(nchunk) * 8));
  if (!starts || !chunks) return fail(DDF_ENOMEM, "device allocation of the BDA block index failed");
  int rc = launch_bda_index(v->bda, v->nblocks, starts, chunks, tmp.st);
  *out = starts;
  return rc;
}

// Mean frequency and wavelength of the channels (gridder.h:164-171): taken from the host fields
// when set, else read back from the device array (a synchronising copy).
int freq_means(const ddf_vis* v, double* fmean, double* wlmean, hipStream_t st) {
  if (v->freq_mean > 0 && v->wavelength_mean > 0) {
    *fmean = v->freq_mean;
    *wlmean = v->wavelength_mean;
    return DDF_OK;
  }
  std::vector<double> f(size_t(v->nchan));
  HIP_TRY(hipMemcpyAsync(f.data(), v->freqs, f.size() * 8, hipMemcpyDeviceToHost, st));
  HIP_TRY(hipStreamSynchronize(st));
  double wl = 0, fm = 0;
  for (double x : f) {
    wl += kC / x;
    fm += x;
  }
  *fmean = fm / double(f.size());
  *wlmean = wl / double(f.size());
  return DDF_OK;
}

// Lanes of a block (log2: 0, 3 or 6), by the mean visibilities per block of a map that covers the chunk and by the
// wavefronts that its blocks give.  Gridding / degridding with Jones of one facet, us with 1, 8 and 64 lanes (maps by
// uvw, and of equal blocks):
//   1 up to 10 visibilities, from 65536 blocks (1024 wavefronts): 287 000 blocks by uvw of 8 460 / 245, 475 / 278,
//     1386 / 853; 386 000 of 13 862 / 415, 725 / 455, 1878 / 1178; 163 000 of 27 509 / 316, 439 / 296, 978 / 634;
//     126 000 equal ones of 12 182 / 109, 217 / 143, 611 / 415; 25 000 of 4 86 / 71, 67 / 49, 144 / 121
//   64 from 256: 165 000 by uvw of 54 -, 720 / 533, 1091 / 762; 56 000 equal ones of 160 -, 390 / 297, 559 / 488;
//     11 000 of 320 -, 202 / 148, 178 / 132
//   64 where 8 leave most of the GPU idle: 2100 blocks of 640 -, 271 / 201, 103 / 69; 1260 of 1 76 / 62, 34 / 33,
//     31 / 32; 4200 of 24 -, 38 / 35, 54 / 46
int plain_group(const ddf_vis* v) {
  const int64_t mean = v->nrow * v->nchan / std::max<int64_t>(1, v->nblocks);
  if (mean <= 10 && v->nblocks >= 65536) return 0;
  return mean >= 256 || v->nblocks < (mean >= 32 ? 4096 : 2048) ? 6 : 3;
}
// The large blocks of a map in a launch with 1 or 8 lanes a block: those of more than 32 turns of its lanes (8 lanes, 16
// turns 1-20 % slower, 64 turns 5-25 %).  A group that took them itself was what the launch waited for: 18 700 blocks of
// 26 visibilities on average (20 antennas close together), gridded and degridded with Jones 870 / 615 us by eights,
// 224 / 171 by wavefronts, 170 / 135 with the large blocks apart.
void plain_large(const ddf_vis* v, int lg, KParams& p) {
  p.large = INT64_MAX;
  p.large_wgs = 0;
  if (lg == 6 || v->nblocks >= v->nrow * v->nchan) return;
  p.large = int64_t(32) << lg;
  p.large_wgs = unsigned(std::min<int64_t>(1024, (v->nblocks + 255) / 256));
}
unsigned grid_blocks(int64_t nblocks, int lg) {
  const int64_t per = 4 * (kWave >> lg);  // blocks of a workgroup
  int64_t need = (nblocks + per - 1) / per;
  int64_t cap = 256 * 16;
  if (need < 1) need = 1;
  return unsigned(need < cap ? need : cap);
}

template <int READ, int JMODE, typename GT>
void launch_grid_g(const KParams& p, int lg, size_t lds, unsigned nb, hipStream_t st) {
  if (lg == 6) hipLaunchKernelGGL((grid_plain<READ, JMODE, GT, 6>), dim3(nb), dim3(256), lds, st, p);
  else if (lg == 3) hipLaunchKernelGGL((grid_plain<READ, JMODE, GT, 3>), dim3(nb), dim3(256), lds, st, p);
  else hipLaunchKernelGGL((grid_plain<READ, JMODE, GT, 0>), dim3(nb), dim3(256), lds, st, p);
}

template <int READ, int JMODE>
int launch_grid_t(const KParams& p, int grid_f64, int lg, size_t lds, unsigned nb, hipStream_t st) {
  if (grid_f64) launch_grid_g<READ, JMODE, double>(p, lg, lds, nb, st);
  else launch_grid_g<READ, JMODE, float>(p, lg, lds, nb, st);
  return DDF_OK;
}

template <int READ>
int launch_grid_r(const KParams& p, int jmode, int grid_f64, int lg, size_t lds, unsigned nb, hipStream_t st) {
  if (jmode == 1) return launch_grid_t<READ, 1>(p, grid_f64, lg, lds, nb, st);
  if (jmode == 2) return launch_grid_t<READ, 2>(p, grid_f64, lg, lds, nb, st);
  return launch_grid_t<READ, 0>(p, grid_f64, lg, lds, nb, st);
}

template <int NCORR, int JMODE, int LG>
void launch_degrid_l(const KParams& p, unsigned nb, hipStream_t st) {
  if (p.large_wgs) hipLaunchKernelGGL((degrid_plain<NCORR, JMODE, LG, true>), dim3(nb), dim3(256), 0, st, p);
  else hipLaunchKernelGGL((degrid_plain<NCORR, JMODE, LG, false>), dim3(nb), dim3(256), 0, st, p);
}

template <int NCORR, int JMODE>
void launch_degrid_g(const KParams& p, int lg, unsigned nb, hipStream_t st) {
  if (lg == 6) hipLaunchKernelGGL((degrid_plain<NCORR, JMODE, 6, false>), dim3(nb), dim3(256), 0, st, p);
  else if (lg == 3) launch_degrid_l<NCORR, JMODE, 3>(p, nb, st);
  else launch_degrid_l<NCORR, JMODE, 0>(p, nb, st);
}

template <int NCORR>
int launch_degrid_r(const KParams& p, int jmode, int lg, unsigned nb, hipStream_t st) {
  if (jmode == 1) launch_degrid_g<NCORR, 1>(p, lg, nb, st);
  else if (jmode == 2) launch_degrid_g<NCORR, 2>(p, lg, nb, st);
  else launch_degrid_g<NCORR, 0>(p, lg, nb, st);
  return DDF_OK;
}

}  // namespace

namespace ddf {
void set_last_error(const std::string& msg) { g_err = msg; }

// The current device's pool, made at its first use (0: this one has none).
static hipError_t device_pool(hipMemPool_t* pool) {
  static std::mutex mu;
  static hipMemPool_t pools[64] = {};
  *pool = nullptr;
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess || dev < 0 || dev >= 64) return e;
  std::lock_guard<std::mutex> lk(mu);
  if (!pools[dev]) {
    hipMemPoolProps props;
    std::memset(&props, 0, sizeof(props));
    props.allocType = hipMemAllocationTypePinned;
    props.location.type = hipMemLocationTypeDevice;
    props.location.id = dev;
    hipMemPool_t made = nullptr;
    e = hipMemPoolCreate(&made, &props);
    if (e != hipSuccess) return e;
    uint64_t keep = kPoolKeep;
    e = hipMemPoolSetAttribute(made, hipMemPoolAttrReleaseThreshold, &keep);
    if (e != hipSuccess) {
      (void)hipMemPoolDestroy(made);
      return e;
    }
    pools[dev] = made;
  }
  *pool = pools[dev];
  return hipSuccess;
}

hipError_t pool_alloc(void** p, size_t bytes, hipStream_t st) {
  hipMemPool_t pool;
  hipError_t e = device_pool(&pool);
  if (e != hipSuccess) return e;
  if (!pool) return hipMallocAsync(p, bytes, st);
  e = hipMallocFromPoolAsync(p, bytes, pool, st);
  if (e == hipSuccess) return e;
  (void)hipGetLastError();
  (void)hipStreamSynchronize(st);
  (void)hipMemPoolTrimTo(pool, 0);
  return hipMallocFromPoolAsync(p, bytes, pool, st);
}

hipError_t pool_trim(size_t keep) {
  hipMemPool_t pool;
  const hipError_t e = device_pool(&pool);
  return e != hipSuccess || !pool ? e : hipMemPoolTrimTo(pool, keep);
}
}  // namespace ddf

// ---- Briggs transform without allocation ------------------------------------------------------
// The per-workgroup partial sums of the robust transform live in a file-scope device array, one
// copy per GPU, instead of a caller workspace: for callers that cannot allocate (graph capture,
// serving loops).  Its address on each device comes from hipGetSymbolAddress, once per device
// (ddf_init, or the first call on a device); host code uses that address, never the symbol.
constexpr int kBriggsBlocks = 256;  // workgroups per band of the robust transform
constexpr int kBriggsMaxBands = 64;
static __device__ __align__(256) double scratch[kBriggsMaxBands * kBriggsBlocks * 2];

namespace {
constexpr int kMaxDevices = 64;
std::mutex g_scratch_mu;
double* g_scratch_ptr[kMaxDevices] = {};

// Address of `scratch` on the current device (resolved once per device).
int scratch_address(double** out) {
  int dev = 0;
  HIP_TRY(hipGetDevice(&dev));
  if (dev < 0 || dev >= kMaxDevices) return fail(DDF_EINVAL, "device index out of range for the scratch table");
  std::lock_guard<std::mutex> lk(g_scratch_mu);
  if (!g_scratch_ptr[dev]) {
    void* ptr = nullptr;
    HIP_TRY(hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch)));
    if (!ptr) return fail(DDF_EHIP, "hipGetSymbolAddress returned a null scratch address");
    g_scratch_ptr[dev] = static_cast<double*>(ptr);
  }
  *out = g_scratch_ptr[dev];
  return DDF_OK;
}
}  // namespace

extern "C" {

int ddf_version(void) { return DDF_ABI_VERSION; }

const char* ddf_last_error(void) { return g_err.c_str(); }

int ddf_init(int device) {
  HIP_TRY(hipSetDevice(device));
  HIP_TRY(hipFree(nullptr));
  double* ptr = nullptr;
  return scratch_address(&ptr);
}

int ddf_bda_index(const int32_t* bda, int64_t bda_len, int64_t nblocks, int64_t* out, void* stream) {
  if (!bda || !out || nblocks < 0 || 2 + nblocks > bda_len) return fail(DDF_EINVAL, "inconsistent BDA map");
  hipStream_t st = static_cast<hipStream_t>(stream);
  Temp tmp(st);
  int64_t nchunk = (nblocks + kScanChunk - 1) / kScanChunk;
  int64_t* chunks = nchunk ? static_cast<int64_t*>(tmp.get(size_t(nchunk) * 8)) : nullptr;
  if (nchunk && !chunks) return fail(DDF_ENOMEM, "device allocation failed");
  return launch_bda_index(bda, nblocks, out, chunks, st);
}

int ddf_grid(const ddf_grid_desc* g, const ddf_vis* v, const ddf_facet* f, void* stream) {
  int rc = check_common(g, v, f);
  if (rc) return rc;
  if (!v->weights || !f->sumwt) return fail(DDF_EINVAL, "weights / sumwt pointer is null");
  if (f->jones.enabled && (!f->jones.sum_jones || !f->jones.sum_jones_chan))
    return fail(DDF_EINVAL, "SumJones / SumJonesChan pointer is null");
  StokesMap sm;
  rc = grid_map(v, &sm);
  if (rc) return rc;
  if (v->nblocks == 0 || v->nrow == 0) return DDF_OK;
  hipStream_t st = static_cast<hipStream_t>(stream);
  double fmean0 = 0, wl_mean = 0;
  rc = freq_means(v, &fmean0, &wl_mean, st);
  if (rc) return rc;
  Temp tmp(st);
  const int64_t* starts = nullptr;
  rc = resolve_block_index(v, tmp, &starts);
  if (rc) return rc;
  KParams p;
  fill_params(p, g, v, f, sm, starts, fmean0, wl_mean);
  const int jmode = f->jones.enabled ? f->jones.mode : 0;
  size_t lds_base = size_t(g->nband) * g->npol + 2 * size_t(g->nband);
  p.chan_lds = (jmode != 0) && (lds_base + 2 * size_t(v->nchan)) * 8 <= 48 * 1024;
  size_t lds = (lds_base + (p.chan_lds ? 2 * size_t(v->nchan) : 0)) * 8;
  if (lds > 60 * 1024) return fail(DDF_EINVAL, "nband * npol too large for the gridding accumulators");
  const int lg = plain_group(v);
  plain_large(v, lg, p);
  unsigned nb = grid_blocks(v->nblocks, lg) + p.large_wgs;
  if (sm.read == 4) rc = launch_grid_r<4>(p, jmode, g->grid_f64, lg, lds, nb, st);
  else if (sm.read == 2) rc = launch_grid_r<2>(p, jmode, g->grid_f64, lg, lds, nb, st);
  else rc = launch_grid_r<1>(p, jmode, g->grid_f64, lg, lds, nb, st);
  if (rc) return rc;
  HIP_TRY(hipGetLastError());
  return DDF_OK;
}

int ddf_degrid(const ddf_grid_desc* g, const ddf_vis* v, const ddf_facet* f, void* stream) {
  int rc = check_common(g, v, f);
  if (rc) return rc;
  if (g->grid_f64) return fail(DDF_EINVAL, "the degridder reads complex64 grids");
  StokesMap sm;
  rc = degrid_map(v, &sm);
  if (rc) return rc;
  if (sm.nstokes > g->npol) return fail(DDF_EINVAL, "grid has fewer polarisations than the requested Stokes parameters");
  if (v->nblocks == 0 || v->nrow == 0) return DDF_OK;
  hipStream_t st = static_cast<hipStream_t>(stream);
  double fmean0 = 0, wl_mean = 0;
  rc = freq_means(v, &fmean0, &wl_mean, st);
  if (rc) return rc;
  Temp tmp(st);
  const int64_t* starts = nullptr;
  rc = resolve_block_index(v, tmp, &starts);
  if (rc) return rc;
  KParams p;
  fill_params(p, g, v, f, sm, starts, fmean0, wl_mean);
  const int jmode = f->jones.enabled ? f->jones.mode : 0;
  const int lg = plain_group(v);
  plain_large(v, lg, p);
  unsigned nb = grid_blocks(v->nblocks, lg) + p.large_wgs;
  if (v->ncorr == 4) rc = launch_degrid_r<4>(p, jmode, lg, nb, st);
  else if (v->ncorr == 2) rc = launch_degrid_r<2>(p, jmode, lg, nb, st);
  else if (v->ncorr == 1) rc = launch_degrid_r<1>(p, jmode, lg, nb, st);
  else return fail(DDF_EINVAL, "ncorr must be 1, 2 or 4");
  if (rc) return rc;
  HIP_TRY(hipGetLastError());
  return DDF_OK;
}

}  // extern "C"

// ---- weights scatter-add ---------------------------------------------------------------------
namespace {
__global__ __launch_bounds__(256) void accumulate_weights(double* grid, int64_t glen, const float* w, const int64_t* idx,
                                                          int64_t n) {
  for (int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x; i < n; i += int64_t(gridDim.x) * blockDim.x) {
    float x = w[i];
    if (x != 0) {
      int64_t k = idx[i];
      if (k >= 0 && k < glen) atomicAdd(&grid[k], double(x));
    }
  }
}
}  // namespace

extern "C" int ddf_accumulate_weights(double* grid, int64_t grid_len, const float* weights, const int64_t* index,
                                      int64_t n, void* stream) {
  if (n < 0 || grid_len < 0) return fail(DDF_EINVAL, "negative size");
  if (n == 0) return DDF_OK;
  if (!grid || !weights || !index) return fail(DDF_EINVAL, "null pointer");
  int64_t nb = (n + 255) / 256;
  if (nb > 65536) nb = 65536;
  hipLaunchKernelGGL(accumulate_weights, dim3(unsigned(nb)), dim3(256), 0, static_cast<hipStream_t>(stream), grid,
                     grid_len, weights, index, n);
  HIP_TRY(hipGetLastError());
  return DDF_OK;
}

// ---- imaging weights: uv-grid index, Briggs transform, renormalisation ---------------------------
namespace {
constexpr double kLightSpeedWeights = 299792458.0;  // ClassVisServer._cc

// One thread per (row, channel): the uv-grid cell of ClassVisServer._uv_to_index
// (ClassVisServer.py:983-1004), in its operation order and without contraction: (u freq) / c, then
// / cell, floored; the int64 cell number is narrowed to int32 as numpy's assignment into an int32
// array does (two's complement), and the band offset added and narrowed again.
__global__ __launch_bounds__(256) void weights_index_k(const double* uvw, const float* w, int64_t nrow, int nchan,
                                                       const double* freqs, const int32_t* chan_band, double cell,
                                                       int64_t npix, int64_t npixx, int nbands, int64_t xymax,
                                                       int32_t* index) {
#pragma clang fp contract(off)
  const int64_t n = nrow * int64_t(nchan);
  for (int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x; i < n; i += int64_t(gridDim.x) * blockDim.x) {
    const int64_t r = i / nchan;
    const int c = int(i - r * nchan);
    double u = uvw[3 * r], v = uvw[3 * r + 1];
    if (v < 0) {
      u = -u;
      v = -v;
    }
    const double f = freqs[c];
    const double ul = (u * f) / kLightSpeedWeights, vl = (v * f) / kLightSpeedWeights;
    const int64_t x = int64_t(floor(ul / cell)) + xymax;
    const int64_t y = int64_t(floor(vl / cell));
    int32_t k = int32_t(uint32_t(uint64_t(y * npixx + x)));
    if (nbands > 1) k = int32_t(uint32_t(uint64_t(int64_t(k) + int64_t(chan_band[c]) * npix)));
    if (w[i] == 0.f) k = 0;
    index[i] = k;
  }
}

// Scatter-add of a [nrow][nchan] weight array through its int32 cell index (the sum of
// pyAccumulateWeightsOntoGrid, GridderSmearPols.cc:32-74, zero weights skipped).  A wavefront takes
// one channel of 64 consecutive rows: rows of one baseline at successive times mostly fall in one
// cell, so the lanes first sum each run of equal cells (segmented scan over the wavefront) and only
// a run's last lane issues the FP64 atomic.
__global__ __launch_bounds__(256) void weights_accumulate_k(double* grid, int64_t glen, const float* w,
                                                            const int32_t* idx, int64_t nrow, int nchan) {
  const int lane = threadIdx.x & 63;
  const int64_t ntile = (nrow + 63) / 64;
  const int64_t ntask = ntile * nchan;
  const int64_t wave0 = (int64_t(blockIdx.x) * blockDim.x + threadIdx.x) >> 6;
  const int64_t nwave = (int64_t(gridDim.x) * blockDim.x) >> 6;
  for (int64_t task = wave0; task < ntask; task += nwave) {
    const int c = int(task % nchan);
    const int64_t r = (task / nchan) * 64 + lane;
    int k = -1;
    double x = 0;
    if (r < nrow) {
      const int64_t i = r * nchan + c;
      const float wi = w[i];
      const int ki = idx[i];
      if (wi != 0.f && ki >= 0 && int64_t(ki) < glen) {
        k = ki;
        x = double(wi);
      }
    }
    // head of this lane's run of equal cells
    const int kp = __shfl_up(k, 1, 64);
    int start = (lane == 0 || kp != k) ? lane : 0;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
      const int o = __shfl_up(start, d, 64);
      if (lane >= d && o > start) start = o;
    }
    // sum from the run's head to this lane
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
      const double y = __shfl_up(x, d, 64);
      if (lane - d >= start) x += y;
    }
    const int kn = __shfl_down(k, 1, 64);
    const bool tail = lane == 63 || kn != k;
    if (tail && k >= 0) atomicAdd(&grid[k], x);
  }
}

// Robust transform of the weight grid (ClassVisServer.py:1188-1197) in two launches over
// kBriggsBlocks workgroups per band: the first writes each workgroup's partial sums of g^2 and g
// over a strided share of the band's cells; the second has every workgroup reduce the band's
// partials in the same order (so each obtains the same avgW = sum g^2 / sum g), then apply
// g <- 1 + g sSq, sSq = num2 / avgW, to its share, the product rounded before the sum.

__global__ __launch_bounds__(256) void weights_briggs_sums_k(const double* grid, int64_t npix, double* part) {
  __shared__ double s2[256], s1[256];
  const int band = blockIdx.y;
  const double* g = grid + int64_t(band) * npix;
  double a2 = 0, a1 = 0;
  for (int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x; i < npix; i += int64_t(gridDim.x) * blockDim.x) {
    const double x = g[i];
    a2 = fma(x, x, a2);
    a1 += x;
  }
  s2[threadIdx.x] = a2;
  s1[threadIdx.x] = a1;
  __syncthreads();
  for (int o = blockDim.x / 2; o > 0; o >>= 1) {
    if (int(threadIdx.x) < o) {
      s2[threadIdx.x] += s2[threadIdx.x + o];
      s1[threadIdx.x] += s1[threadIdx.x + o];
    }
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    part[(int64_t(band) * gridDim.x + blockIdx.x) * 2] = s2[0];
    part[(int64_t(band) * gridDim.x + blockIdx.x) * 2 + 1] = s1[0];
  }
}

__global__ __launch_bounds__(256) void weights_briggs_apply_k(double* grid, int64_t npix, const double* part,
                                                              double num2) {
#pragma clang fp contract(off)
  __shared__ double s2[256], s1[256];
  const int band = blockIdx.y;
  const double* pb = part + int64_t(band) * gridDim.x * 2;
  double a2 = 0, a1 = 0;
  for (int k = threadIdx.x; k < int(gridDim.x); k += blockDim.x) {
    a2 += pb[2 * k];
    a1 += pb[2 * k + 1];
  }
  s2[threadIdx.x] = a2;
  s1[threadIdx.x] = a1;
  __syncthreads();
  for (int o = blockDim.x / 2; o > 0; o >>= 1) {
    if (int(threadIdx.x) < o) {
      s2[threadIdx.x] += s2[threadIdx.x + o];
      s1[threadIdx.x] += s1[threadIdx.x + o];
    }
    __syncthreads();
  }
  const double avg = s2[0] / s1[0];
  const double ssq = num2 / avg;
  double* g = grid + int64_t(band) * npix;
  for (int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x; i < npix; i += int64_t(gridDim.x) * blockDim.x) {
    const double t = g[i] * ssq;
    g[i] = 1. + t;
  }
}

// weights[i] /= grid[index[i]] (ClassVisServer.py:1035-1040): indices >= grid_len read cell 0 as
// the reference sets them; negative ones count from the end as numpy indexing does (below
// -grid_len, where numpy raises, cell 0).  The quotient is formed in FP64 and rounded to FP32, as
// numpy's in-place division of a float32 array by float64 values is.
__global__ __launch_bounds__(256) void weights_finalize_k(float* w, const int32_t* idx, int64_t n, const double* grid,
                                                          int64_t glen) {
  for (int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x; i < n; i += int64_t(gridDim.x) * blockDim.x) {
    int64_t k = idx[i];
    if (k >= glen) k = 0;
    if (k < 0) k += glen;
    if (k < 0) k = 0;
    w[i] = float(double(w[i]) / grid[k]);
  }
}

unsigned weight_blocks(int64_t n) {
  int64_t nb = (n + 255) / 256;
  return unsigned(nb > 65536 ? 65536 : (nb < 1 ? 1 : nb));
}
}  // namespace

extern "C" int ddf_weights_index(const double* uvw, const float* weights, int64_t nrow, int nchan, const double* freqs,
                                 const int32_t* chan_band, double cell, int64_t npix, int64_t npixx, int nbands,
                                 int64_t xymax, int32_t* index, void* stream) {
  if (nrow < 0 || nchan < 0 || nbands < 1) return fail(DDF_EINVAL, "negative size or nbands < 1");
  if (nrow == 0 || nchan == 0) return DDF_OK;
  if (!uvw || !weights || !freqs || !index) return fail(DDF_EINVAL, "null pointer");
  if (nbands > 1 && !chan_band) return fail(DDF_EINVAL, "chan_band is required when nbands > 1");
  if (!(cell > 0)) return fail(DDF_EINVAL, "cell must be positive");
  hipLaunchKernelGGL(weights_index_k, dim3(weight_blocks(nrow * int64_t(nchan))), dim3(256), 0,
                     static_cast<hipStream_t>(stream), uvw, weights, nrow, nchan, freqs, chan_band, cell, npix, npixx,
                     nbands, xymax, index);
  HIP_TRY(hipGetLastError());
  return DDF_OK;
}

extern "C" int ddf_weights_accumulate(double* grid, int64_t grid_len, const float* weights, const int32_t* index,
                                      int64_t nrow, int nchan, void* stream) {
  if (nrow < 0 || nchan < 0 || grid_len < 0) return fail(DDF_EINVAL, "negative size");
  if (nrow == 0 || nchan == 0) return DDF_OK;
  if (!grid || !weights || !index) return fail(DDF_EINVAL, "null pointer");
  const int64_t waves = ((nrow + 63) / 64) * nchan;
  int64_t nb = (waves + 3) / 4;
  if (nb > 65536) nb = 65536;
  hipLaunchKernelGGL(weights_accumulate_k, dim3(unsigned(nb)), dim3(256), 0, static_cast<hipStream_t>(stream), grid,
                     grid_len, weights, index, nrow, nchan);
  HIP_TRY(hipGetLastError());
  return DDF_OK;
}

extern "C" int64_t ddf_weights_briggs_work_size(int nbands) {
  return nbands > 0 ? int64_t(nbands) * kBriggsBlocks * 2 : 0;
}

extern "C" int ddf_weights_briggs(double* grid, int nbands, int64_t npix, double robust, double* work,
                                  int64_t work_len, void* stream) {
  if (nbands < 0 || npix < 0) return fail(DDF_EINVAL, "negative size");
  if (nbands == 0 || npix == 0) return DDF_OK;
  if (nbands > 65535) return fail(DDF_EINVAL, "more than 65535 bands");
  if (!grid || !work) return fail(DDF_EINVAL, "null pointer");
  if (work_len < ddf_weights_briggs_work_size(nbands)) return fail(DDF_EINVAL, "workspace too small");
  // numeratorSqrt = 5 * 10 ** (-Robust); its square as Python's float ** 2 (an exact square, rounded)
  const double num = 5.0 * std::pow(10.0, -robust);
  const double num2 = num * num;
  const dim3 grid2(kBriggsBlocks, unsigned(nbands));
  hipLaunchKernelGGL(weights_briggs_sums_k, grid2, dim3(256), 0, static_cast<hipStream_t>(stream), grid, npix, work);
  HIP_TRY(hipGetLastError());
  hipLaunchKernelGGL(weights_briggs_apply_k, grid2, dim3(256), 0, static_cast<hipStream_t>(stream), grid, npix, work,
                     num2);
  HIP_TRY(hipGetLastError());
  return DDF_OK;
}

extern "C" int ddf_weights_briggs_noalloc(double* grid, int nbands, int64_t npix, double robust, void* stream) {
  if (nbands < 0 || npix < 0) return fail(DDF_EINVAL, "negative size");
  if (nbands > kBriggsMaxBands)
    return fail(DDF_EINVAL, "ddf_weights_briggs_noalloc handles at most 64 bands (use ddf_weights_briggs)");
  if (nbands == 0 || npix == 0) return DDF_OK;
  if (!grid) return fail(DDF_EINVAL, "null pointer");
  double* part = nullptr;
  int rc = scratch_address(&part);
  if (rc) return rc;
  // every partial the second launch reads is written by the first in this call: nothing to clear
  const double num = 5.0 * std::pow(10.0, -robust);
  const double num2 = num * num;
  const dim3 grid2(kBriggsBlocks, unsigned(nbands));
  hipLaunchKernelGGL(weights_briggs_sums_k, grid2, dim3(256), 0, static_cast<hipStream_t>(stream), grid, npix, part);
  HIP_TRY(hipGetLastError());
  hipLaunchKernelGGL(weights_briggs_apply_k, grid2, dim3(256), 0, static_cast<hipStream_t>(stream), grid, npix, part,
                     num2);
  HIP_TRY(hipGetLastError());
  return DDF_OK;
}

extern "C" int ddf_weights_finalize(float* weights, const int32_t* index, int64_t n, const double* grid,
                                    int64_t grid_len, void* stream) {
  if (n < 0 || grid_len < 0) return fail(DDF_EINVAL, "negative size");
  if (n == 0) return DDF_OK;
  if (!weights || !index || !grid || grid_len == 0) return fail(DDF_EINVAL, "null pointer or empty grid");
  hipLaunchKernelGGL(weights_finalize_k, dim3(weight_blocks(n)), dim3(256), 0, static_cast<hipStream_t>(stream), weights,
                     index, n, grid, grid_len);
  HIP_TRY(hipGetLastError());
  return DDF_OK;
}

// ---- chunk flag preparation (ClassMS.py:1155-1167) -------------------------------------------------
namespace {
// One thread per (row, channel): autocorrelation rows flagged, NaN visibilities (either part)
// flagged, the values flagged so far overwritten with 1e9 + 0i, then every correlation flagged when
// any is, in the reference's order.
__global__ __launch_bounds__(256) void prepare_flags_k(uint8_t* flags, float2* data, const int32_t* a0,
                                                       const int32_t* a1, int64_t nrow, int nchan, int ncorr,
                                                       int vec4) {
  const int64_t n = nrow * int64_t(nchan);
  if (vec4) {
    // four correlations with 4-byte aligned flags and 16-byte aligned values: the flags of a
    // (row, channel) as one 32-bit word, the values as two 16-byte loads
    uint32_t* fw = reinterpret_cast<uint32_t*>(flags);
    float4* d4 = reinterpret_cast<float4*>(data);
    for (int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x; i < n; i += int64_t(gridDim.x) * blockDim.x) {
      const int64_t r = i / nchan;
      const bool autoc = a0[r] == a1[r];
      const uint32_t f0 = fw[i];
      bool f[4];
#pragma unroll
      for (int k = 0; k < 4; ++k) f[k] = ((f0 >> (8 * k)) & 0xFFu) != 0 || autoc;
      if (data) {
        float4 x0 = d4[2 * i], x1 = d4[2 * i + 1];
        f[0] = f[0] || isnan(x0.x) || isnan(x0.y);
        f[1] = f[1] || isnan(x0.z) || isnan(x0.w);
        f[2] = f[2] || isnan(x1.x) || isnan(x1.y);
        f[3] = f[3] || isnan(x1.z) || isnan(x1.w);
        if (f[0] || f[1]) {
          if (f[0]) { x0.x = 1e9f; x0.y = 0.f; }
          if (f[1]) { x0.z = 1e9f; x0.w = 0.f; }
          d4[2 * i] = x0;
        }
        if (f[2] || f[3]) {
          if (f[2]) { x1.x = 1e9f; x1.y = 0.f; }
          if (f[3]) { x1.z = 1e9f; x1.w = 0.f; }
          d4[2 * i + 1] = x1;
        }
      }
      const bool any = f[0] || f[1] || f[2] || f[3];
      fw[i] = any ? 0x01010101u : 0u;
    }
    return;
  }
  for (int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x; i < n; i += int64_t(gridDim.x) * blockDim.x) {
    const int64_t r = i / nchan;
    const bool autoc = a0[r] == a1[r];
    bool any = false;
    for (int k = 0; k < ncorr; ++k) {
      const int64_t j = i * ncorr + k;
      bool f = flags[j] != 0 || autoc;
      if (data) {
        const float2 x = data[j];
        f = f || isnan(x.x) || isnan(x.y);
        if (f) data[j] = make_float2(1e9f, 0.f);
      }
      any = any || f;
      flags[j] = f ? 1 : 0;
    }
    if (any)
      for (int k = 0; k < ncorr; ++k) flags[i * ncorr + k] = 1;
  }
}
}  // namespace

extern "C" int ddf_prepare_flags(uint8_t* flags, float* data, const int32_t* a0, const int32_t* a1, int64_t nrow,
                                 int nchan, int ncorr, void* stream) {
  if (nrow < 0 || nchan < 0 || ncorr < 1 || ncorr > 4) return fail(DDF_EINVAL, "bad sizes (ncorr must be 1..4)");
  if (nrow == 0 || nchan == 0) return DDF_OK;
  if (!flags || !a0 || !a1) return fail(DDF_EINVAL, "null pointer");
  const int vec4 = ncorr == 4 && reinterpret_cast<uintptr_t>(flags) % 4 == 0 &&
                   reinterpret_cast<uintptr_t>(data) % 16 == 0;
  hipLaunchKernelGGL(prepare_flags_k, dim3(weight_blocks(nrow * int64_t(nchan))), dim3(256), 0,
                     static_cast<hipStream_t>(stream), flags, reinterpret_cast<float2*>(data), a0, a1, nrow, nchan,
                     ncorr, vec4);
  HIP_TRY(hipGetLastError());
  return DDF_OK;
}

// ======================================================================================================
// Batched plan (host side).
// ======================================================================================================
struct ddf_plan {
  BatchParams pg, pd, pa;         // gridding, degridding, and the adjoint of degrid pass A with its own items
  VisP vg, vd;
  FacetDev* d_facets = nullptr;
  int32_t* d_support = nullptr;
  // pair codes (0x80 | band for a placed (block, facet) record) read by the cycle passes
  uint8_t* pcode_g = nullptr;
  uint8_t* pcode_d = nullptr;
  uint32_t* recs_g = nullptr;
  uint32_t* recs_d = nullptr;
  uint64_t* bstamp_g = nullptr;  // stamp records in bin order (tile offset, support, CF offset)
  float* slots_g = nullptr;      // one LDS tile image per grid work item (null: atomic flush)
  uint32_t* tile_first_g = nullptr;
  uint32_t* tile_count_g = nullptr;
  uint32_t* live_g = nullptr;    // count, then the tiles that have slots in reach
  uint64_t* bstamp_d = nullptr;
  BinItem* items_g = nullptr;
  BinItem* items_d = nullptr;
  BinItem* items_a = nullptr;
  float2* V = nullptr;
  float2* M = nullptr;
  DegridRuns deg = {};            // degrid visibility list: runs share a block and a Jones key
  RunList runs = {};              // grid pass A on runs (entry null: grid_pass_a)
  unsigned nwg_runs = 0;
  // work-queue counters (kQueueStride words apart): [0] grid pass A, [1, 9) grid pass B (one per item range), [9, 17) degrid
  // pass A, [17] the adjoint of degrid pass B, [18, 26) the adjoint of degrid pass A
  // [kQueueRuns ...) grid pass A on runs, one per facet group
  static constexpr int kQueueRuns = 2 + 3 * kItemRanges, kQueues = kQueueRuns + kRunQueues;
  uint32_t* queues = nullptr;
  uint32_t* queue(int k) const { return queues + k * kQueueStride; }
  const float2* jsrc[2] = {nullptr, nullptr};  // caller's DD / beam Jones tables
  double2* jprep[2] = {nullptr, nullptr};      // prepared copies (JonesP::pk / pb)
  float2* jprepf[2] = {nullptr, nullptr};      // complex64 prepared copies (JonesP::pkf / pbf)
  unsigned nwg = 0;
  unsigned nwg_tiles[3] = {0, 0, 0};  // tile passes (grid B, degrid A, adjoint): as many as fit
  int64_t stats[8] = {0, 0, 0, 0, 0, 0, 0, 0};
  PoolArena arena;
  hipStream_t st = nullptr;       // the stream of the build
  // per-pass timing (ddf_plan_timing): events around each pass on the launch stream
  int timing = 0;
  hipEvent_t ev[DDF_PLAN_NPASS][2] = {};
  int ev_set[DDF_PLAN_NPASS] = {};
  ~ddf_plan() {
    arena.close();  // (a cycle may still be under way on any stream)
    for (auto& e : ev)
      for (hipEvent_t x : e)
        if (x) (void)hipEventDestroy(x);
  }
  void mark(int pass, int end, hipStream_t st) {
    if (!timing) return;
    (void)hipEventRecord(ev[pass][end], st);
    if (end) ev_set[pass] = 1;
  }
  template <typename T>
  T* alloc(size_t n) {
    return static_cast<T*>(arena.get(std::max<size_t>(n, 1) * sizeof(T), st));
  }
};

namespace {

int prepare_jones(ddf_plan* P, hipStream_t st) {
  for (int k = 0; k < 2; ++k)
    if (P->jprep[k] && batched_prepare_jones(P->pg, P->jsrc[k], P->jprep[k], P->jprepf[k], k == 0, st)) return DDF_EHIP;
  return DDF_OK;
}

int fill_vis(VisP& out, const ddf_vis* v, const int64_t* starts) {
  std::memset(&out, 0, sizeof(out));
  out.vis = reinterpret_cast<float2*>(v->vis);
  out.uvw = v->uvw;
  out.flags = v->flags;
  out.weights = v->weights;
  out.freqs = v->freqs;
  out.chan_map = v->chan_map;
  out.nrow = v->nrow;
  out.nchan = v->nchan;
  out.ncorr = v->ncorr;
  out.bda = v->bda;
  out.bda_start = starts;
  out.nblocks = v->nblocks;
  out.bda_len = v->bda_len;
  out.sparse = v->sparsification;
  out.equi = v->chan_equidistant && v->nchan > 1;
  return DDF_OK;
}

void fill_batch(BatchParams& p, const ddf_grid_desc* g, const ddf_facet* f0, const StokesMap& sm,
                double fmean0, double wl_mean) {
  std::memset(&p, 0, sizeof(p));
  p.nband = g->nband;
  p.npol = g->npol;
  p.ny = g->ny;
  p.nx = g->nx;
  p.incr0 = g->incr[0];
  p.incr1 = g->incr[1];
  p.nw = f0->cf.nw;
  p.overs = f0->cf.overs;
  p.ref_wave = f0->cf.ref_wave;
  p.wmax = f0->cf.wmax;
  p.nstokes = sm.nstokes;
  p.read = sm.read;
  std::memcpy(p.sm, sm.m, sizeof(p.sm));
  const ddf_jones& j = f0->jones;
  p.jmode = j.enabled ? j.mode : 0;
  p.jp.enabled = j.enabled;
  p.jp.mode = j.mode;
  p.jp.interp = j.interp_mode;
  p.jp.kms = reinterpret_cast<const float2*>(j.kms);
  p.jp.beam = reinterpret_cast<const float2*>(j.beam);
  for (int i = 0; i < 4; ++i) {
    p.jp.kdims[i] = j.kms_dims[i];
    p.jp.bdims[i] = j.beam_dims[i];
  }
  p.jp.ktime = j.kms_time;
  p.jp.kchan = j.kms_chan;
  p.jp.btime = j.beam_time;
  p.jp.bchan = j.beam_chan;
  p.jp.a0 = j.a0;
  p.jp.a1 = j.a1;
  p.jp.coefs = j.coefs;
  p.jp.ncoefs = j.coefs ? j.ncoefs : 0;
  p.jp.apply_amp = j.apply_amp;
  p.jp.apply_phase = j.apply_phase;
  p.jp.scale = j.scale_jones;
  p.jp.calib_error = j.calib_error;
  p.dp.enabled = f0->decorr.enabled;
  p.dp.tsmear = f0->decorr.tsmear;
  p.dp.fsmear = f0->decorr.fsmear;
  p.dp.uvw_dt = f0->decorr.uvw_dt;
  p.dp.dt = f0->decorr.dt;
  p.dp.dnu = f0->decorr.dnu;
  p.dp.fscale = decorr_fscale(f0->decorr.dnu);
  p.fmean0 = fmean0;
  p.tscale0 = decorr_tscale(fmean0);
  p.wl_mean = wl_mean;
}

// The work items of a map: of each tile's records (their counts by CF-plane group in hg) up to `chunk` an item.
struct TileItems {
  std::vector<BinItem> items;               // in launch order
  std::vector<uint32_t> packs, range;       // see BatchParams
  std::vector<int64_t> start;               // first record of each tile
  std::vector<uint32_t> first, count;       // first slot and slots of each tile
  int64_t records = 0;
  int nranges = 1;
};
// A tile's sub-bins (CF planes) are split into ngrp groups of consecutive planes, each chunked into
// items.  Slots are numbered tile by tile (a tile's slots consecutive, for grid_slot_reduce); the launch order
// is (facet, band, plane group, tile), so that the workgroups running at one time read the CF planes
// of one group and those stay in L2.
TileItems tile_items(const BatchParams& p, std::vector<uint32_t> hg, int64_t ngrp, int chunk, int64_t light) {
  TileItems L;
  const int64_t ntile_fb = int64_t(p.ntiles_x) * p.ntiles_y, ntile_all = int64_t(p.nf) * p.nband * ntile_fb;
  // A tile of up to `light` records is one item: its groups' counts go to the first group (121 facets x 4 bands:
  // 506 000 items of 37 records otherwise, each with a tile to clear and a slot to write).
  const int64_t whole = std::min<int64_t>(chunk, light);
  for (int64_t i = 0; i < ntile_all; ++i) {
    uint32_t* h = &hg[size_t(i * ngrp)];
    int64_t all = 0;
    for (int64_t g = 0; g < ngrp; ++g) all += h[g];
    if (all > whole) continue;
    std::fill(h, h + ngrp, 0u);
    h[0] = uint32_t(all);
  }
  // tile-major pass: each tile's first record and first slot, each (tile, group)'s item count
  L.start.resize(size_t(ntile_all));
  L.first.resize(size_t(ntile_all));
  L.count.resize(size_t(ntile_all));
  int64_t nitem = 0;
  for (int64_t i = 0; i < ntile_all; ++i) {
    L.start[size_t(i)] = L.records;
    L.first[size_t(i)] = uint32_t(nitem);
    for (int64_t g = 0; g < ngrp; ++g) {
      const int64_t cg = hg[size_t(i * ngrp + g)];
      L.records += cg;
      nitem += (cg + chunk - 1) / chunk;
    }
    L.count[size_t(i)] = uint32_t(nitem - L.first[size_t(i)]);
  }
  if (L.records >= (int64_t(1) << 32)) return L;  // (refused by the caller)
  L.items.reserve(size_t(nitem));
  for (int64_t fb = 0; fb < int64_t(p.nf) * p.nband; ++fb) {
    for (int64_t g = 0; g < ngrp; ++g) {
      for (int64_t tin = 0; tin < ntile_fb; ++tin) {
        const int64_t i = fb * ntile_fb + tin;
        const int64_t cg = hg[size_t(i * ngrp + g)];
        if (cg == 0) continue;
        int64_t g0 = 0, s0 = 0;  // records and items of the tile's earlier groups
        for (int64_t h = 0; h < g; ++h) {
          const int64_t ch = hg[size_t(i * ngrp + h)];
          g0 += ch;
          s0 += (ch + chunk - 1) / chunk;
        }
        for (int64_t b = 0, c = 0; b < cg; b += chunk, ++c) {
          BinItem it;
          it.begin = uint32_t(L.start[size_t(i)] + g0 + b);
          it.end = uint32_t(L.start[size_t(i)] + g0 + (b + chunk < cg ? b + chunk : cg));
          it.facet = int16_t(fb / p.nband);
          it.band = int16_t(fb % p.nband);
          it.tx = int16_t(tin % p.ntiles_x);
          it.ty = int16_t(tin / p.ntiles_x);
          it.slot = uint32_t(L.first[size_t(i)] + s0 + c);
          L.items.push_back(it);
        }
      }
    }
  }
  // packs of consecutive items
  const std::vector<BinItem>& items = L.items;
  const size_t pack_items = std::min<size_t>(kPackItems, std::max<size_t>(1, items.size() / 16384));
  L.packs.reserve(items.size() / pack_items + 2);
  for (size_t k = 0; k < items.size();) {
    L.packs.push_back(uint32_t(k));
    uint32_t n = 0;
    for (size_t k0 = k; k < items.size() && k - k0 < pack_items && n < kPackRecords; ++k) n += items[k].end - items[k].begin;
  }
  const uint32_t npacks = uint32_t(L.packs.size());
  L.packs.push_back(uint32_t(items.size()));
  // kItemRanges contiguous ranges of the launch order with about equal record counts: the
  // workgroups of one XCD take the packs of their own range first, so the items in flight on an
  // XCD come from few (facet, plane group)s and their CF planes stay in that XCD's L2.  Only with
  // many items: with few, the heaviest items (neighbouring uv tiles) would share one XCD's CUs, so
  // all items then form one range.
  L.nranges = items.size() >= kRangeMinItems ? kItemRanges : 1;
  L.range.assign(size_t(L.nranges) + 1, npacks);
  L.range[0] = 0;
  if (L.nranges > 1) {
    int64_t acc = 0;
    int x = 1;
    for (uint32_t k = 0; k < npacks && x < L.nranges; ++k) {
      for (uint32_t i = L.packs[k]; i < L.packs[k + 1]; ++i) acc += int64_t(items[i].end) - items[i].begin;
      while (x < L.nranges && acc * L.nranges >= L.records * x) L.range[size_t(x++)] = k + 1;
    }
  }
  return L;
}

// The items, packs and ranges on the device, and what of them the passes read from p.
int upload_items(ddf_plan* P, BatchParams& p, const TileItems& L, BinItem** items_out, hipStream_t st) {
  BinItem* d_items = P->alloc<BinItem>(L.items.size());
  uint32_t* d_range = P->alloc<uint32_t>(L.range.size());
  uint32_t* d_packs = P->alloc<uint32_t>(L.packs.size());
  if (!d_items || !d_range || !d_packs) return fail(DDF_ENOMEM, "plan allocation failed");
  if (!L.items.empty())
    HIP_TRY(hipMemcpyAsync(d_items, L.items.data(), L.items.size() * sizeof(BinItem), hipMemcpyHostToDevice, st));
  HIP_TRY(hipMemcpyAsync(d_range, L.range.data(), L.range.size() * 4, hipMemcpyHostToDevice, st));
  HIP_TRY(hipMemcpyAsync(d_packs, L.packs.data(), L.packs.size() * 4, hipMemcpyHostToDevice, st));
  p.pack_range = d_range;
  p.pack_first = d_packs;
  p.npacks = uint32_t(L.packs.size()) - 1;
  p.nranges = L.nranges;
  p.nitems_b = uint32_t(L.items.size());
  p.tile_records = L.records;
  *items_out = d_items;
  return DDF_OK;
}

// Count -> scan -> fill of the valid records, then the work items (largest first).  adj: the items of
// the adjoint pass over the same records (null: none).
int build_bins(ddf_plan* P, BatchParams& p, const VisP& v, const uint64_t* place, int chunk, uint32_t** recs_out,
               BinItem** items_out, int64_t* nrec, bool stamp_order, hipStream_t st, uint32_t** tile_first_out,
               uint32_t** tile_count_out, BatchParams* adj, BinItem** adj_items_out) {
  const int64_t nsub = 2 * int64_t(p.nw);  // CF-plane sub-bins of each tile
  const int64_t ntile_all = int64_t(p.nf) * p.nband * p.ntiles_y * p.ntiles_x;
  const int64_t nbins = ntile_all * nsub;
  Temp scratch(st);  // not needed by the cycle
  uint32_t* counts = scratch.get<uint32_t>(size_t(nbins));
  uint32_t* fill = scratch.get<uint32_t>(size_t(nbins));
  int64_t* bstart = scratch.get<int64_t>(size_t(nbins));
  const int64_t ngrp = nsub < 4 ? nsub : 4;
  uint32_t* gcount = scratch.get<uint32_t>(size_t(ntile_all * ngrp));
  int64_t* tstart = scratch.get<int64_t>(size_t(ntile_all));
  if (!counts || !fill || !bstart || !gcount || !tstart) return fail(DDF_ENOMEM, "plan allocation failed");
  HIP_TRY(hipMemsetAsync(counts, 0, size_t(nbins) * 4, st));
  HIP_TRY(hipMemsetAsync(fill, 0, size_t(nbins) * 4, st));
  if (batched_count(p, v.nblocks, place, counts, st)) return fail(DDF_EHIP, "plan_count launch failed");
  // only the (tile, group) counts come to the host; the bin starts are formed on the device
  if (batched_group_counts(counts, ntile_all, int(nsub), int(ngrp), gcount, st))
    return fail(DDF_EHIP, "plan_group_counts launch failed");
  std::vector<uint32_t> hg(static_cast<size_t>(ntile_all * ngrp));
  HIP_TRY(hipMemcpyAsync(hg.data(), gcount, hg.size() * 4, hipMemcpyDeviceToHost, st));
  HIP_TRY(hipStreamSynchronize(st));
  // Records of an item: those asked for, or 2048, down to 64 where a plan has too few to give every
  // wavefront of the tile passes an item (9 facets of 189^2, 11 000 records: a wavefront with a heavy
  // tile's 1000 records took longer than all others together).
  const int most = chunk > 0 ? chunk : 2048;
  if (chunk <= 0) {
    int64_t all = 0;
    for (uint32_t c : hg) all += c;
    chunk = int(std::min<int64_t>(most, std::max<int64_t>(64, all / 4096 / 64 * 64)));
  }
  const TileItems L = tile_items(p, hg, ngrp, chunk, kWholeTileRecords);
  const int64_t tot = L.records;
  if (tot >= (int64_t(1) << 32)) return fail(DDF_EINVAL, "too many (block, facet) records for one plan");
  HIP_TRY(hipMemcpyAsync(tstart, L.start.data(), L.start.size() * 8, hipMemcpyHostToDevice, st));
  if (batched_bin_starts(counts, tstart, ntile_all, int(nsub), bstart, st))
    return fail(DDF_EHIP, "plan_bin_starts launch failed");
  uint32_t* recs = P->alloc<uint32_t>(size_t(tot));
  if (!recs) return fail(DDF_ENOMEM, "plan allocation failed");
  BinItem* d_items = nullptr;
  int rc = upload_items(P, p, L, &d_items, st);
  if (rc) return rc;
  if (tile_first_out) {
    uint32_t* tf = P->alloc<uint32_t>(size_t(ntile_all));
    uint32_t* tc = P->alloc<uint32_t>(size_t(ntile_all));
    if (!tf || !tc) return fail(DDF_ENOMEM, "plan allocation failed");
    HIP_TRY(hipMemcpyAsync(tf, L.first.data(), size_t(ntile_all) * 4, hipMemcpyHostToDevice, st));
    HIP_TRY(hipMemcpyAsync(tc, L.count.data(), size_t(ntile_all) * 4, hipMemcpyHostToDevice, st));
    *tile_first_out = tf;
    *tile_count_out = tc;
  }
  if (batched_fill(p, v.nblocks, place, bstart, fill, recs, st)) return fail(DDF_EHIP, "plan_fill launch failed");
  // the records are sorted within the larger items; where the adjoint has items of its own, the others
  // are parts of them
  BinItem* sort_items = d_items;
  uint32_t nsort = p.nitems_b;
  TileItems A;
  if (adj) {
    // The adjoint adds in FP32 both in an item's tile and, by atomics, in the grids: a cell's error grows with
    // the items of its tile (with 64 records each the gradients of dense small plans came out three times as far
    // from 64 bits) and with the records of an item (tiles of 512 records taken whole: 1.4 times).  So its items
    // are a plane group's 2048 records: 25 facets x 4 bands, 5.64 ms a gradient, 5.61 with tiles taken
    // whole, 6.00 with FP64 tiles.
    *adj = p;
    A = tile_items(p, hg, ngrp, most, 0);
    rc = upload_items(P, *adj, A, adj_items_out, st);
    if (rc) return rc;
    sort_items = *adj_items_out;
    nsort = adj->nitems_b;
  }
  if (batched_sort_items(p, place, recs, tot, sort_items, nsort, stamp_order, st))
    return fail(DDF_EHIP, "sorting the records of the work items failed");
  HIP_TRY(hipStreamSynchronize(st));
  *recs_out = recs;
  *items_out = d_items;
  *nrec = tot;
  return DDF_OK;
}

}  // namespace

namespace {

// The run list of the grid map, for grid_pass_a_runs.  It is left out where a plan does not take it or where its
// 8 bytes a visibility cannot be had: grid_pass_a grids the map then.
int build_runs(ddf_plan* P, const ddf_vis* v, int group, hipStream_t st) {
  RunList rl = {};
  if (!batched_runs_layout(P->pg, P->vg, group, &rl)) return DDF_OK;
  const int64_t nb = v->nblocks;
  Temp rt(st), list(st);
  auto leave = [] {
    (void)hipGetLastError();
    return int(DDF_OK);
  };
  int32_t* cnt = rt.get<int32_t>(size_t(nb));
  int64_t* tmp = rt.get<int64_t>(size_t((nb + kScanChunk - 1) / kScanChunk));
  int64_t* start = list.get<int64_t>(size_t(nb) + 1);
  if (!cnt || !tmp || !start) return leave();
  if (batched_vis_counts(P->vg, cnt, st)) return fail(DDF_EHIP, "launch failed");
  int rc = launch_scan(cnt, nb, 0, start, tmp, st);
  if (rc) return rc;
  int64_t last_start = 0;
  int32_t last_cnt = 0;
  if (hipMemcpyAsync(&last_start, start + nb - 1, 8, hipMemcpyDeviceToHost, st) != hipSuccess ||
      hipMemcpyAsync(&last_cnt, cnt + nb - 1, 4, hipMemcpyDeviceToHost, st) != hipSuccess ||
      hipStreamSynchronize(st) != hipSuccess)
    return fail(DDF_EHIP, "copy failed");
  const int64_t total = last_start + last_cnt;
  batched_run_split(total, &rl);
  uint64_t* entry = list.get<uint64_t>(size_t(total));
  uint32_t* item = list.get<uint32_t>(size_t(rl.nitems) + 1);
  if (!entry || !item) return leave();
  rl.start = start;
  if (hipMemcpyAsync(start + nb, &total, 8, hipMemcpyHostToDevice, st) != hipSuccess ||
      hipStreamSynchronize(st) != hipSuccess || batched_run_entries(P->pg, P->vg, start, entry, st) ||
      batched_run_items(P->vg, rl, item, st))
    return fail(DDF_EHIP, "launch failed");
  rl.item = item;
  rl.entry = entry;
  P->runs = rl;
  P->arena.take(list.arena);
  return DDF_OK;
}

}  // namespace

extern "C" int ddf_plan_create(const ddf_grid_desc* g, const ddf_vis* vgrid, const ddf_vis* vdegrid,
                               const ddf_facet* facets, void* const* models, int32_t nfacets,
                               const ddf_plan_opts* opts, ddf_plan** out, void* stream) {
  if (!out) return fail(DDF_EINVAL, "null plan output");
  *out = nullptr;
  if (nfacets <= 0 || !facets || !models) return fail(DDF_EINVAL, "no facets");
  int rc = check_common(g, vgrid, &facets[0]);
  if (rc) return rc;
  rc = check_common(g, vdegrid, &facets[0]);
  if (rc) return rc;
  if (g->grid_f64) return fail(DDF_EINVAL, "the batched path accumulates complex64 grids");
  if (g->nx >= 65536 || g->ny >= 65536 || g->nband >= 128) return fail(DDF_EINVAL, "grid too large for the plan records");
  if (!vgrid->weights) return fail(DDF_EINVAL, "weights pointer is null");
  const ddf_cf& c0 = facets[0].cf;
  if (2 * c0.nw > 255 || c0.overs > 255) return fail(DDF_EINVAL, "too many w-planes / oversampling for the plan records");
  StokesMap smg, smd;
  rc = grid_map(vgrid, &smg);
  if (rc) return rc;
  rc = degrid_map(vdegrid, &smd);
  if (rc) return rc;
  if (smd.nstokes > g->npol) return fail(DDF_EINVAL, "grid has fewer polarisations than the requested Stokes parameters");
  if ((vgrid->nblocks + 1) * int64_t(nfacets) >= (int64_t(1) << 32) ||
      (vdegrid->nblocks + 1) * int64_t(nfacets) >= (int64_t(1) << 32))
    return fail(DDF_EINVAL, "blocks x facets exceeds the 32-bit record index");
  hipStream_t st = static_cast<hipStream_t>(stream);
  // shared CF geometry: every facet's supports and plane offsets read back together
  for (int i = 1; i < nfacets; ++i) {
    const ddf_cf& ci = facets[i].cf;
    if (ci.nw != c0.nw || ci.overs != c0.overs || ci.ref_wave != c0.ref_wave || ci.wmax != c0.wmax)
      return fail(DDF_EINVAL, "all facets of a plan must share nw, OverS, RefWave and wmax");
    if (!ci.data || !ci.offset || !ci.support) return fail(DDF_EINVAL, "bad CF table");
    if (!facets[i].grid || !models[i] || !facets[i].sumwt) return fail(DDF_EINVAL, "facet buffer is null");
    if (facets[0].jones.enabled && (!facets[i].jones.sum_jones || !facets[i].jones.sum_jones_chan))
      return fail(DDF_EINVAL, "SumJones buffers are null");
  }
  const size_t nw0 = size_t(c0.nw);
  std::vector<int32_t> sups(size_t(nfacets) * nw0);
  std::vector<int64_t> offs(size_t(nfacets) * 2 * nw0);
  {
    Temp ct(st);
    std::vector<CfSource> src(static_cast<size_t>(nfacets));
    for (int i = 0; i < nfacets; ++i) src[size_t(i)] = CfSource{facets[i].cf.support, facets[i].cf.offset};
    CfSource* d_src = static_cast<CfSource*>(ct.get(src.size() * sizeof(CfSource)));
    int32_t* d_sup = static_cast<int32_t*>(ct.get(sups.size() * 4));
    int64_t* d_off = static_cast<int64_t*>(ct.get(offs.size() * 8));
    if (!d_src || !d_sup || !d_off) return fail(DDF_ENOMEM, "plan allocation failed");
    HIP_TRY(hipMemcpyAsync(d_src, src.data(), src.size() * sizeof(CfSource), hipMemcpyHostToDevice, st));
    if (batched_cf_info(d_src, nfacets, c0.nw, d_sup, d_off, st)) return fail(DDF_EHIP, "reading the CF tables failed");
    HIP_TRY(hipMemcpyAsync(sups.data(), d_sup, sups.size() * 4, hipMemcpyDeviceToHost, st));
    HIP_TRY(hipMemcpyAsync(offs.data(), d_off, offs.size() * 8, hipMemcpyDeviceToHost, st));
    HIP_TRY(hipStreamSynchronize(st));
  }
  const std::vector<int32_t> sup0(sups.begin(), sups.begin() + c0.nw);
  int maxsup = 0;
  for (int32_t x : sup0) {
    if (x <= 0 || x % 2 == 0) return fail(DDF_EINVAL, "CF supports must be odd and positive");
    maxsup = x > maxsup ? x : maxsup;
  }
  for (int i = 1; i < nfacets; ++i)
    if (!std::equal(sup0.begin(), sup0.end(), sups.begin() + size_t(i) * nw0))
      return fail(DDF_EINVAL, "all facets of a plan must share the CF supports");
  if (!models[0] || !facets[0].sumwt) return fail(DDF_EINVAL, "facet buffer is null");
  if (facets[0].jones.enabled && (!facets[0].jones.sum_jones || !facets[0].jones.sum_jones_chan))
    return fail(DDF_EINVAL, "SumJones buffers are null");

  ddf_plan* P = new ddf_plan();
  P->st = st;
  auto bail = [&](int code) {
    delete P;
    return code;
  };
  double fm = 0, wl = 0;
  rc = freq_means(vgrid, &fm, &wl, st);
  if (rc) return bail(rc);
  fill_batch(P->pg, g, &facets[0], smg, fm, wl);
  fill_batch(P->pd, g, &facets[0], smd, fm, wl);
  P->pg.dopsf = g->dopsf;
  // prepared Jones tables (FP64, facet-fastest), refreshed from the caller's tables at every
  // grid / degrid call so that new Jones values need no new plan
  for (int k = 0; k < 2; ++k) {
    const ddf_jones& j = facets[0].jones;
    const float* src = k ? j.beam : j.kms;
    const int32_t* dims = k ? j.beam_dims : j.kms_dims;
    if (!j.enabled || !src) continue;
    const size_t n = size_t(dims[0]) * dims[1] * dims[2] * dims[3] * 4;
    double2* dst = P->alloc<double2>(n);
    float2* dstf = P->alloc<float2>(n);
    if (!dst || !dstf) return bail(fail(DDF_ENOMEM, "plan allocation failed"));
    P->jsrc[k] = reinterpret_cast<const float2*>(src);
    P->jprep[k] = dst;
    P->jprepf[k] = dstf;
    for (BatchParams* bp : {&P->pg, &P->pd}) {
      if (k) {
        bp->jp.pb = dst;
        bp->jp.pbf = dstf;
      } else {
        bp->jp.pk = dst;
        bp->jp.pkf = dstf;
      }
    }
  }
  if (prepare_jones(P, st)) return bail(fail(DDF_EHIP, "Jones preparation failed"));
  ddf_plan_opts o{};
  if (opts) o = *opts;
  const int tile = o.tile > 0 ? o.tile : 16;
  const int chunk = o.chunk;
  const int halo = (maxsup - 1) / 2;
  {
    // the tile passes hold one (T + 2 h)^2 complex64 image per polarisation in LDS
    int dev = 0, lds_max = 0;
    if (hipGetDevice(&dev) != hipSuccess ||
        hipDeviceGetAttribute(&lds_max, hipDeviceAttributeMaxSharedMemoryPerBlock, dev) != hipSuccess)
      return bail(fail(DDF_EHIP, "device query failed"));
    const int W = tile + 2 * halo;
    const int np = std::max(std::min(smg.nstokes, g->npol), smd.nstokes);
    if (size_t(np) * W * W * 8 + 4096 > size_t(lds_max))
      return bail(fail(DDF_EINVAL, "uv tile too large for LDS at this support and polarisation count"));
    // stamp records hold the tile offset in 16 bits and the support in 5
    if (W > 255 || maxsup > 31) return bail(fail(DDF_EINVAL, "uv tile or CF support too large for the stamp records"));
    // ... and the oversampled sub-kernel index in 11 bits
    if (int64_t(c0.overs) * c0.overs > 0x7FF) return bail(fail(DDF_EINVAL, "CF oversampling too large for the stamp records"));
  }
  int G = o.group;
  if (G <= 0) {
    int ng = (nfacets + 31) / 32;
    G = (nfacets + ng - 1) / ng;
  }
  if (G > 64) G = 64;  // gridding pass A aligns its slots (G lanes each) to wavefronts
  // facet descriptors
  P->d_support = P->alloc<int32_t>(sup0.size());
  if (!P->d_support || hipMemcpyAsync(P->d_support, sup0.data(), sup0.size() * 4, hipMemcpyHostToDevice, st) != hipSuccess)
    return bail(fail(DDF_EHIP, "plan upload failed"));
  // padded copies of the facets' CF planes for degrid pass A (rows of an even pitch, plane pl at twice its
  // offset), all in one buffer, each at an even element
  std::vector<size_t> pad(size_t(nfacets) + 1, 0);
  for (int i = 0; i < nfacets; ++i) {
    int64_t total = 0, total_pad = 0;
    for (int pl = 0; pl < 2 * c0.nw; ++pl) {
      const int64_t S = sup0[size_t(pl < c0.nw ? pl : pl - c0.nw)], O2 = int64_t(c0.overs) * c0.overs;
      const int64_t off = offs[size_t(i) * 2 * nw0 + size_t(pl)];
      total = std::max(total, off + O2 * S * S);
      total_pad = std::max(total_pad, 2 * off + O2 * S * (S + (S & 1)));
    }
    // grid pass B addresses a facet's CF values by a 32-bit byte offset
    if (total * int64_t(sizeof(float2)) >= (int64_t(1) << 32))
      return bail(fail(DDF_EINVAL, "a facet's CF table reaches 4 GiB"));
    pad[size_t(i) + 1] = pad[size_t(i)] + size_t(total_pad + (total_pad & 1));
  }
  float2* padded = P->alloc<float2>(pad.back());
  if (!padded) return bail(fail(DDF_ENOMEM, "plan allocation failed"));
  std::vector<FacetDev> hf(static_cast<size_t>(nfacets));
  for (int i = 0; i < nfacets; ++i) {
    const ddf_facet& f = facets[i];
    FacetDev& d = hf[size_t(i)];
    d.cft = padded + pad[size_t(i)];
    d.grid = f.grid;
    d.model = models[i];
    d.cf = reinterpret_cast<const float2*>(f.cf.data);
    d.cf_offset = f.cf.offset;
    d.cu = f.cu;
    d.cv = f.cv;
    d.l0 = f.l0;
    d.m0 = f.m0;
    d.n0 = std::sqrt(1 - f.l0 * f.l0 - f.m0 * f.m0) - 1;
    d.dec_l0 = f.decorr.l0;
    d.dec_m0 = f.decorr.m0;
    d.kms_dir = f.jones.kms_dir;
    d.beam_dir = f.jones.beam_dir;
    d.sumwt = f.sumwt;
    d.sum_jones = f.jones.sum_jones;
    d.sum_jones_chan = f.jones.sum_jones_chan;
  }
  P->d_facets = P->alloc<FacetDev>(hf.size());
  P->queues = P->alloc<uint32_t>(ddf_plan::kQueues * kQueueStride);
  if (!P->d_facets || !P->queues) return bail(fail(DDF_ENOMEM, "plan allocation failed"));
  if (hipMemcpyAsync(P->d_facets, hf.data(), hf.size() * sizeof(FacetDev), hipMemcpyHostToDevice, st) != hipSuccess)
    return bail(fail(DDF_EHIP, "plan upload failed"));
  if (batched_cf_pad(P->d_facets, nfacets, P->d_support, c0.nw, c0.overs, maxsup, st))
    return bail(fail(DDF_EHIP, "CF copy launch failed"));
  for (BatchParams* bp : {&P->pg, &P->pd}) {
    bp->facets = P->d_facets;
    bp->nf = nfacets;
    bp->support = P->d_support;
    bp->prec = o.precision;
    bp->tile = tile;
    bp->halo = halo;
    bp->ntiles_x = (g->nx + tile - 1) / tile;
    bp->ntiles_y = (g->ny + tile - 1) / tile;
    bp->group = G;
    bp->slots = 256 / G;
    bp->ngroups = (nfacets + G - 1) / G;
  }
  P->pd.jmode = vdegrid == vgrid ? P->pg.jmode : P->pd.jmode;
  // block indices of both maps
  const int64_t* sg = vgrid->bda_start;
  const int64_t* sd = vdegrid->bda_start;
  for (int k = 0; k < 2; ++k) {
    const ddf_vis* v = k ? vdegrid : vgrid;
    const int64_t*& s = k ? sd : sg;
    if (s || v->nblocks == 0) continue;
    Temp scratch(st);
    int64_t* ns = P->alloc<int64_t>(size_t(v->nblocks));
    int64_t* tmp = scratch.get<int64_t>(size_t((v->nblocks + kScanChunk - 1) / kScanChunk));
    if (!ns || !tmp) return bail(fail(DDF_ENOMEM, "plan allocation failed"));
    rc = launch_bda_index(v->bda, v->nblocks, ns, tmp, st);
    if (rc) return bail(rc);
    s = ns;
  }
  fill_vis(P->vg, vgrid, sg);
  fill_vis(P->vd, vdegrid, sd);
  // per-block descriptors of the grid map (grid pass A reads them instead of the row lists)
  if (vgrid->bda_len >= (int64_t(1) << 32) || vgrid->nchan > 65535)
    return bail(fail(DDF_EINVAL, "BDA map too long or too many channels for the block descriptors"));
  {
    uint4* d = P->alloc<uint4>(size_t(vgrid->nblocks));
    if (!d) return bail(fail(DDF_ENOMEM, "plan allocation failed"));
    if (vgrid->nblocks && batched_block_desc(P->vg, d, st)) return bail(fail(DDF_EHIP, "plan_block_desc failed"));
    P->vg.bdesc = d;
  }
  P->pg.nblk = vgrid->nblocks;
  P->pd.nblk = vdegrid->nblocks;
  // first frequency and step of equidistant channels (the anchors of ChanPhasor)
  for (VisP* pv : {&P->vg, &P->vd}) {
    if (!pv->equi) continue;
    double f2[2] = {0, 0};
    if (hipMemcpyAsync(f2, pv->freqs, sizeof(f2), hipMemcpyDeviceToHost, st) != hipSuccess ||
        hipStreamSynchronize(st) != hipSuccess)
      return bail(fail(DDF_EHIP, "reading the channel frequencies failed"));
    pv->f0 = f2[0];
    pv->df = f2[1] - f2[0];
  }
  // placements
  // (of both maps, while the plan is built: ddf_plan_placements recomputes them)
  Temp scratch_g(st), scratch_d(st);
  uint64_t* place_g = scratch_g.get<uint64_t>(size_t(vgrid->nblocks) * nfacets);
  uint64_t* place_d = scratch_d.get<uint64_t>(size_t(vdegrid->nblocks) * nfacets);
  if (!place_g || !place_d) return bail(fail(DDF_ENOMEM, "plan allocation failed"));
  if (vgrid->nblocks && batched_place(P->pg, P->vg, false, place_g, st)) return bail(fail(DDF_EHIP, "plan_place failed"));
  if (vdegrid->nblocks && batched_place(P->pd, P->vd, true, place_d, st)) return bail(fail(DDF_EHIP, "plan_place failed"));
  // bins
  int64_t nr = 0;
  rc = build_bins(P, P->pg, P->vg, place_g, chunk, &P->recs_g, &P->items_g, &nr, true, st, &P->tile_first_g, &P->tile_count_g,
                  nullptr, nullptr);
  if (rc) return bail(rc);
  const uint32_t ni = P->pg.nitems_b;
  P->stats[0] = nr;
  P->stats[2] = ni;
  P->bstamp_g = P->alloc<uint64_t>(size_t(nr));
  if (!P->bstamp_g || batched_stamp_records(P->pg, place_g, P->recs_g, nr, P->bstamp_g, st))
    return bail(fail(DDF_ENOMEM, "plan allocation failed"));
  // the grid map's placements reduced to pair codes (3.5 GB -> 0.44 GB at the 81-facet chunk)
  {
    const size_t np = size_t(vgrid->nblocks) * nfacets;
    P->pcode_g = P->alloc<uint8_t>(np);
    if (!P->pcode_g || batched_pair_codes(place_g, int64_t(np), P->pcode_g, st) ||
        hipStreamSynchronize(st) != hipSuccess)
      return bail(fail(DDF_ENOMEM, "plan allocation failed"));
    scratch_g.free();
  }

  {
    // tile slots of the gridding items (plain stores + a deterministic reduction instead of
    // global atomics); without the memory for them the tiles are flushed with atomics
    const int W = tile + 2 * halo;
    const int npg = smg.nstokes < g->npol ? smg.nstokes : g->npol;
    const size_t n = size_t(ni) * size_t(npg) * 2 * size_t(W) * size_t(W);
    if (ni) {
      P->slots_g = P->alloc<float>(n);
      if (P->slots_g) P->live_g = P->alloc<uint32_t>(1 + size_t(nfacets) * g->nband * P->pg.ntiles_y * P->pg.ntiles_x);
      if (!P->live_g) {
        P->slots_g = nullptr;
        (void)hipGetLastError();
      } else if (batched_live_tiles(P->pg, P->tile_count_g, P->live_g, st)) {
        return bail(fail(DDF_EHIP, "launch failed"));
      }
    }
  }
  rc = build_bins(P, P->pd, P->vd, place_d, chunk, &P->recs_d, &P->items_d, &nr, false, st, nullptr, nullptr, &P->pa, &P->items_a);
  if (rc) return bail(rc);
  P->stats[1] = nr;
  P->stats[3] = P->pd.nitems_b;
  P->bstamp_d = P->alloc<uint64_t>(size_t(nr));
  if (!P->bstamp_d || batched_stamp_records(P->pd, place_d, P->recs_d, nr, P->bstamp_d, st))
    return bail(fail(DDF_ENOMEM, "plan allocation failed"));
  {
    const size_t np = size_t(vdegrid->nblocks) * nfacets;
    P->pcode_d = P->alloc<uint8_t>(np);
    if (!P->pcode_d || batched_pair_codes(place_d, int64_t(np), P->pcode_d, st) ||
        hipStreamSynchronize(st) != hipSuccess)
      return bail(fail(DDF_ENOMEM, "plan allocation failed"));
    scratch_d.free();
  }

  // pass A layout
  const int64_t bpi = o.blocks_per_item > 0 ? o.blocks_per_item : 128;
  P->pg.blocks_per_item = bpi;
  P->pg.nchunks = (vgrid->nblocks + bpi - 1) / bpi;
  if (int64_t(P->pg.ngroups) * P->pg.nchunks >= (int64_t(1) << 32)) return bail(fail(DDF_EINVAL, "too many work items"));
  P->pg.nitems_a = uint32_t(int64_t(P->pg.ngroups) * P->pg.nchunks);
  P->pd.blocks_per_item = bpi;
  P->pd.nchunks = (vdegrid->nblocks + bpi - 1) / bpi;
  if (int64_t(P->pd.ngroups) * P->pd.nchunks >= (int64_t(1) << 32)) return bail(fail(DDF_EINVAL, "too many work items"));
  P->pd.nitems_a = uint32_t(int64_t(P->pd.ngroups) * P->pd.nchunks);
  const size_t per_f = size_t(g->nband) * g->npol + 2 * size_t(g->nband);
  if (size_t(nfacets) * per_f * 8 > 40 * 1024) return bail(fail(DDF_EINVAL, "facets x bands too large for one plan"));
  // pass A LDS: per-facet sums, visibility staging, and (when they fit in 80 KB with the rest,
  // so that two workgroups share a compute unit) the group's per-channel Jones sums
  const size_t stage_bytes = batched_grid_a_stage_bytes(G, P->pg.read);
  P->pg.chan_lds = (P->pg.jmode != 0) &&
                   (size_t(nfacets) * per_f + size_t(G) * (2 * size_t(vgrid->nchan) + 1)) * 8 + stage_bytes <= 80 * 1024;
  if (size_t(nfacets) * per_f * 8 + stage_bytes > 80 * 1024)
    return bail(fail(DDF_EINVAL, "facets x bands too large for one plan"));
  // LDS tiles
  const int W = tile + 2 * halo;
  const int npg = smg.nstokes < g->npol ? smg.nstokes : g->npol;
  if (size_t(npg > smd.nstokes ? npg : smd.nstokes) * W * W * 8 > 64 * 1024)
    return bail(fail(DDF_EINVAL, "tile too large for LDS: lower opts.tile"));
  // record values
  P->V = P->alloc<float2>(size_t(vgrid->nblocks) * nfacets * smg.nstokes);
  P->M = P->alloc<float2>(size_t(vdegrid->nblocks) * nfacets * smd.nstokes);
  if (!P->V || !P->M) return bail(fail(DDF_ENOMEM, "plan allocation failed"));
  if (hipMemsetAsync(P->M, 0, size_t(vdegrid->nblocks) * nfacets * smd.nstokes * 8, st) != hipSuccess)
    return bail(fail(DDF_EHIP, "memset failed"));
  // visibility list of the degrid map
  Temp rt(st);
  int64_t* vs = nullptr;
  if (vdegrid->nblocks) {
    int32_t* cnt = rt.get<int32_t>(size_t(vdegrid->nblocks));
    vs = rt.get<int64_t>(size_t(vdegrid->nblocks));
    int64_t* tmp = rt.get<int64_t>(size_t((vdegrid->nblocks + kScanChunk - 1) / kScanChunk));
    if (!cnt || !vs || !tmp) return bail(fail(DDF_ENOMEM, "plan allocation failed"));
    if (batched_vis_counts(P->vd, cnt, st)) return bail(fail(DDF_EHIP, "launch failed"));
    rc = launch_scan(cnt, vdegrid->nblocks, 0, vs, tmp, st);
    if (rc) return bail(rc);
    int64_t last_start = 0;
    int32_t last_cnt = 0;
    if (hipMemcpyAsync(&last_start, vs + vdegrid->nblocks - 1, 8, hipMemcpyDeviceToHost, st) != hipSuccess ||
        hipMemcpyAsync(&last_cnt, cnt + vdegrid->nblocks - 1, 4, hipMemcpyDeviceToHost, st) != hipSuccess ||
        hipStreamSynchronize(st) != hipSuccess)
      return bail(fail(DDF_EHIP, "copy failed"));
    P->deg.nvl = last_start + last_cnt;
  }
  if (P->deg.nvl > 0) {  // (blocks without visibilities leave nothing to list)
    DegridRuns& d = P->deg;
    uint64_t* vrc = P->alloc<uint64_t>(size_t(d.nvl));
    uint32_t* vblk = P->alloc<uint32_t>(size_t(d.nvl));
    if (!vrc || !vblk) return bail(fail(DDF_ENOMEM, "plan allocation failed"));
    d.vrc = vrc;
    d.vblk = vblk;
    if (batched_vlist(P->vd, vs, vrc, vblk, st)) return bail(fail(DDF_EHIP, "launch failed"));
    // runs of consecutive entries with one block and one Jones key: degrid pass B forms each
    // facet's Jones product once per run
    if (d.nvl >= (int64_t(1) << 32)) return bail(fail(DDF_EINVAL, "degrid visibility list too long for one plan"));
    int32_t* flag = static_cast<int32_t*>(rt.get(size_t(d.nvl) * sizeof(int32_t)));
    int64_t* excl = static_cast<int64_t*>(rt.get(size_t(d.nvl) * sizeof(int64_t)));
    int64_t* ctmp = static_cast<int64_t*>(rt.get(size_t((d.nvl + kScanChunk - 1) / kScanChunk) * sizeof(int64_t)));
    if (!flag || !excl || !ctmp) return bail(fail(DDF_ENOMEM, "plan allocation failed"));
    if (batched_run_ids(P->pd, P->vd, vrc, vblk, d.nvl, flag, nullptr, nullptr, nullptr, 0, st))
      return bail(fail(DDF_EHIP, "launch failed"));
    // exclusive scan of n counts and the total
    auto scan_total = [&](const int32_t* x, int64_t n, int64_t* out, int64_t* total) {
      int rs = launch_scan(x, n, 0, out, ctmp, st);
      if (rs) return rs;
      int64_t last = 0;
      int32_t own = 0;
      if (hipMemcpyAsync(&last, out + n - 1, 8, hipMemcpyDeviceToHost, st) != hipSuccess ||
          hipMemcpyAsync(&own, x + n - 1, 4, hipMemcpyDeviceToHost, st) != hipSuccess ||
          hipStreamSynchronize(st) != hipSuccess)
        return fail(DDF_EHIP, "copy failed");
      *total = last + own;
      return int(DDF_OK);
    };
    rc = scan_total(flag, d.nvl, excl, &d.nruns);
    if (rc) return bail(rc);
    uint32_t* run_first = P->alloc<uint32_t>(size_t(d.nruns));
    if (!run_first) return bail(fail(DDF_ENOMEM, "plan allocation failed"));
    d.run_first = run_first;
    if (batched_run_ids(P->pd, P->vd, vrc, vblk, d.nvl, flag, excl, nullptr, run_first, 1, st))
      return bail(fail(DDF_EHIP, "launch failed"));
    const bool jones = P->pd.jmode != 0;
    // (no fewer quads than runs, nor than a fourth of the visibilities)
    if (batched_quads_take(P->pd) && quads_pay(d.nvl, d.nruns, std::max(d.nruns, (d.nvl + 3) / 4), nfacets, jones)) {
      int32_t* cnt4 = static_cast<int32_t*>(rt.get(size_t(d.nruns) * sizeof(int32_t)));
      int64_t* first4 = static_cast<int64_t*>(rt.get(size_t(d.nruns) * sizeof(int64_t)));
      if (!cnt4 || !first4) return bail(fail(DDF_ENOMEM, "plan allocation failed"));
      if (batched_quad_counts(d, cnt4, st)) return bail(fail(DDF_EHIP, "launch failed"));
      rc = scan_total(cnt4, d.nruns, first4, &d.nquads);
      if (rc) return bail(rc);
      if (quads_pay(d.nvl, d.nruns, d.nquads, nfacets, jones)) {
        uint32_t* run_quad = P->alloc<uint32_t>(size_t(d.nruns));
        uint32_t* quad_run = P->alloc<uint32_t>(size_t((d.nquads + 63) / 64));
        uint8_t* fold = P->alloc<uint8_t>(size_t((d.nvl + 255) / 256));
        if (!run_quad || !quad_run || !fold) return bail(fail(DDF_ENOMEM, "plan allocation failed"));
        if (batched_quads(d, cnt4, first4, run_quad, quad_run, st) ||
            batched_fold(flag, excl, d.nvl, nfacets, fold, st))
          return bail(fail(DDF_EHIP, "launch failed"));
        d.fold = fold;
        d.run_quad = run_quad;
        d.quad_run = quad_run;
      }
    }
    if (!d.run_quad) {
      uint32_t* vrun = P->alloc<uint32_t>(size_t(d.nvl));
      if (!vrun) return bail(fail(DDF_ENOMEM, "plan allocation failed"));
      d.vrun = vrun;
      if (batched_run_ids(P->pd, P->vd, vrc, vblk, d.nvl, flag, excl, vrun, nullptr, 1, st))
        return bail(fail(DDF_EHIP, "launch failed"));
    }
  }
  P->stats[4] = P->deg.nvl;
  P->stats[6] = tile;
  P->stats[7] = G;
  int dev = 0;
  hipDeviceProp_t prop;
  if (hipGetDevice(&dev) != hipSuccess || hipGetDeviceProperties(&prop, dev) != hipSuccess)
    return bail(fail(DDF_EHIP, "device query failed"));
  P->nwg = unsigned(o.workgroups > 0 ? o.workgroups : prop.multiProcessorCount * 4);
  P->nwg_runs = unsigned(o.workgroups > 0 ? o.workgroups : prop.multiProcessorCount);
  P->pd.tile_threads = 256;
  if (o.workgroups > 0) {
    for (unsigned& x : P->nwg_tiles) x = unsigned(o.workgroups);
  } else if (batched_tile_wgs(P->pg, P->pd, P->nwg_tiles)) {
    return bail(fail(DDF_EHIP, "occupancy query failed"));
  }
  // (last: everything else comes before its memory)
  rc = build_runs(P, vgrid, o.group, st);
  if (rc) return bail(rc);
  if (hipStreamSynchronize(st) != hipSuccess) return bail(fail(DDF_EHIP, "plan build failed"));
  *out = P;
  return DDF_OK;
}

extern "C" int ddf_plan_grid(ddf_plan* P, float* vis, int32_t dopsf, void* stream) {
  if (!P) return fail(DDF_EINVAL, "null plan");
  hipStream_t st = static_cast<hipStream_t>(stream);
  VisP v = P->vg;
  if (vis) v.vis = reinterpret_cast<float2*>(vis);
  BatchParams p = P->pg;
  p.dopsf = dopsf;
  if (prepare_jones(P, st)) return fail(DDF_EHIP, "Jones preparation failed");
  if (batched_reset(P->queue(0), 1 + kItemRanges, st)) return fail(DDF_EHIP, "launch failed");
  if (P->runs.entry && batched_reset(P->queue(ddf_plan::kQueueRuns), P->runs.ngroups, st)) return fail(DDF_EHIP, "launch failed");
  P->mark(DDF_PASS_GRID_A, 0, st);
  if (P->runs.entry) {
    if (batched_grid_runs(p, v, P->runs, P->pcode_g, P->V, P->queue(ddf_plan::kQueueRuns), P->nwg_runs, st))
      return fail(DDF_EHIP, "grid pass A launch failed");
  } else
  if (p.nitems_a && batched_grid_a(p, v, P->pcode_g, P->V, P->queue(0), P->nwg, st)) return fail(DDF_EHIP, "grid pass A launch failed");
  P->mark(DDF_PASS_GRID_A, 1, st);
  P->mark(DDF_PASS_GRID_B, 0, st);
  if (p.nitems_b && batched_grid_b(p, P->bstamp_g, P->V, P->items_g, P->recs_g, P->queue(1), P->nwg_tiles[0], P->slots_g,
                                     P->tile_first_g, P->tile_count_g, P->live_g, st))
    return fail(DDF_EHIP, "grid pass B launch failed");
  P->mark(DDF_PASS_GRID_B, 1, st);
  return DDF_OK;
}

extern "C" int ddf_plan_degrid(ddf_plan* P, float* vis, void* stream) {
  if (!P) return fail(DDF_EINVAL, "null plan");
  hipStream_t st = static_cast<hipStream_t>(stream);
  VisP v = P->vd;
  if (vis) v.vis = reinterpret_cast<float2*>(vis);
  if (prepare_jones(P, st)) return fail(DDF_EHIP, "Jones preparation failed");
  if (batched_reset(P->queue(1 + kItemRanges), kItemRanges, st)) return fail(DDF_EHIP, "launch failed");
  P->mark(DDF_PASS_DEGRID_A, 0, st);
  if (P->pd.nitems_b && batched_degrid_a(P->pd, P->bstamp_d, P->M, P->items_d, P->recs_d, P->queue(1 + kItemRanges), P->nwg_tiles[1], st))
    return fail(DDF_EHIP, "degrid pass A launch failed");
  P->mark(DDF_PASS_DEGRID_A, 1, st);
  P->mark(DDF_PASS_DEGRID_B, 0, st);
  if (batched_degrid_b(P->pd, v, P->M, P->deg, st))
    return fail(DDF_EHIP, "degrid pass B launch failed");
  P->mark(DDF_PASS_DEGRID_B, 1, st);
  return DDF_OK;
}

extern "C" int ddf_plan_degrid_adjoint(ddf_plan* P, const float* vis_bar, void* stream) {
  if (!P || !vis_bar) return fail(DDF_EINVAL, "null argument");
  hipStream_t st = static_cast<hipStream_t>(stream);
  if (prepare_jones(P, st)) return fail(DDF_EHIP, "Jones preparation failed");
  if (batched_reset(P->queue(1 + 2 * kItemRanges), 1 + kItemRanges, st)) return fail(DDF_EHIP, "launch failed");
  const float2* vb = reinterpret_cast<const float2*>(vis_bar);
  P->mark(DDF_PASS_ADJ_B, 0, st);
  if (P->pd.nitems_a && batched_degrid_b_adjoint(P->pd, P->vd, P->pcode_d, vb, P->M, P->queue(1 + 2 * kItemRanges), P->nwg, st))
    return fail(DDF_EHIP, "degrid adjoint pass B launch failed");
  P->mark(DDF_PASS_ADJ_B, 1, st);
  P->mark(DDF_PASS_ADJ_A, 0, st);
  if (P->pa.nitems_b && batched_degrid_a_adjoint(P->pa, P->bstamp_d, P->M, P->items_a, P->recs_d, P->queue(2 + 2 * kItemRanges), P->nwg_tiles[2], st))
    return fail(DDF_EHIP, "degrid adjoint pass A launch failed");
  P->mark(DDF_PASS_ADJ_A, 1, st);
  return DDF_OK;
}

extern "C" int ddf_plan_info(const ddf_plan* P, int64_t* out, int32_t n) {
  if (!P || !out) return fail(DDF_EINVAL, "null argument");
  for (int i = 0; i < n && i < 8; ++i) out[i] = i == 5 ? int64_t(P->arena.bytes()) : P->stats[i];
  for (int i = 8; i < n && i < 11; ++i) out[i] = int64_t(P->nwg_tiles[i - 8]);
  return DDF_OK;
}

extern "C" int ddf_plan_placements(const ddf_plan* P, int32_t degrid, uint64_t* out, int64_t n, void* stream) {
  if (!P || !out) return fail(DDF_EINVAL, "null argument");
  const BatchParams& p = degrid ? P->pd : P->pg;
  const int64_t nb = degrid ? P->vd.nblocks : P->vg.nblocks;
  const int64_t need = nb * int64_t(p.nf);
  if (n < need) return fail(DDF_EINVAL, "output holds fewer than nblocks * nfacets records");
  if (need == 0) return DDF_OK;
  // recomputed into out (the plan keeps only the pair codes): the same kernel on the same inputs
  if (batched_place(p, degrid ? P->vd : P->vg, degrid != 0, out, static_cast<hipStream_t>(stream)))
    return fail(DDF_EHIP, "plan_place failed");
  return DDF_OK;
}

extern "C" int ddf_plan_timing(ddf_plan* P, int32_t enable) {
  if (!P) return fail(DDF_EINVAL, "null plan");
  if (enable && !P->ev[0][0]) {
    for (auto& e : P->ev)
      for (hipEvent_t& x : e) HIP_TRY(hipEventCreate(&x));
  }
  P->timing = enable ? 1 : 0;
  return DDF_OK;
}

extern "C" int ddf_plan_pass_ms(ddf_plan* P, float* ms, int32_t n) {
  if (!P || !ms) return fail(DDF_EINVAL, "null argument");
  for (int i = 0; i < n; ++i) {
    ms[i] = -1.f;
    if (i >= DDF_PLAN_NPASS || !P->ev_set[i]) continue;
    HIP_TRY(hipEventSynchronize(P->ev[i][1]));
    HIP_TRY(hipEventElapsedTime(&ms[i], P->ev[i][0], P->ev[i][1]));
  }
  return DDF_OK;
}

extern "C" int ddf_trim_memory(void) {
  HIP_TRY(hipDeviceSynchronize());
  HIP_TRY(pool_trim(0));
  return DDF_OK;
}

extern "C" int ddf_plan_destroy(ddf_plan* P) {
  delete P;
  return DDF_OK;
}
