// Baseline-dependent-averaging (BDA) block maps built on the device, in the reference int32 word
// format (DDFacet/Data/ClassSmearMapping.py:83-135):
//   [NTot_lo, NTot_hi, size_0 .. size_{NTot-1}, rec_0, rec_1, ...],  rec_b = [chStart, chEnd, rows...]
// with the per-baseline block lists concatenated in lexicographic order of the string key
// "a0:a1" (ClassSmearMapping.py:113) and each baseline's rows in increasing row order
// (np.where((A0 == a0) & (A1 == a1)), :498).
//
// Steps (the reference runs one process-pool job per baseline, ClassSmearMapping.py:64-79):
//   keys     per row the rank of its baseline's string key (a host table), autocorrelations last
//   sort     stable radix sort of the rows by that rank: each baseline's rows become contiguous, in
//            row order
//   segments first / last sorted position of every baseline
//   count    one wavefront per baseline walks its rows (the builder's sequential scan: time blocks
//            cut on the accumulated |duvw| or the phase, channel blocks from the block's smallest
//            decorrelation span) and counts blocks and words
//   scan     exclusive sums over the baselines in key order -> block and word offsets
//   walk     the same walk again, writing one descriptor per block
//   emit     one thread per block writes its size word and record
// The builder's FP64 arithmetic is evaluated in the reference's operation order with
// contraction off, so every cut and every channel boundary equals the host builder's.
#include <hip/hip_runtime.h>
#include <hipcub/hipcub.hpp>

#include <cmath>
#include <cstring>
#include <string>
#include <vector>

#include "../../include/ddfgpu.h"
#include "ddf_pool.h"

namespace ddf {
void set_last_error(const std::string& msg);  // ddfgpu.hip: the message ddf_last_error() returns
}

namespace {

int bfail(int code, const std::string& m) {
  ddf::set_last_error(m);
  return code;
}

struct BlockDesc {
  int64_t word;    // offset of the record inside the records region
  int64_t row0;    // first sorted-row position of the block
  int32_t nrows;
  int32_t ch0, ch1;
  int32_t pad;
};

struct BdaParams {
  int32_t mode;
  int32_t nchan;
  int32_t nbl;
  // mode 1 (GiveBlocksRowsListBL_old, ClassSmearMapping.py:496-625)
  double duv_cut;  // C dPhi / (pi l nu0)
  double k_dnu;    // (C / pi) dPhi
  double l;
  double dfreq;
  // mode 2 (GiveBlocksRowsListBL as restated in ddfacet_amd/bda.py)
  double k_phase;  // 2 pi nu0 / C
  double lmax, nmax;
  double k_span;   // (C / (2 pi)) dPhi
  double dphi;
  int32_t per_row;  // C dPhi / (2 pi nu0) == 0: every row its own time block
};

__global__ void bda_keys_k(const int32_t* a0, const int32_t* a1, int64_t nrow, const int32_t* rank, int na, int nbl,
                           uint32_t* keys, uint32_t* rows) {
  for (int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x; i < nrow; i += int64_t(gridDim.x) * blockDim.x) {
    const int p = a0[i], q = a1[i];
    uint32_t k = uint32_t(nbl);
    if (p != q && p >= 0 && q >= 0 && p < na && q < na) k = uint32_t(rank[p * na + q]);
    keys[i] = k;
    rows[i] = uint32_t(i);
  }
}

__global__ void bda_fill64_k(int64_t* x, int64_t n, int64_t v) {
  for (int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x; i < n; i += int64_t(gridDim.x) * blockDim.x) x[i] = v;
}

// seg[2 k] = first sorted position of baseline k, seg[2 k + 1] = one past its last (0, 0: absent)
__global__ void bda_segments_k(const uint32_t* keys, int64_t nrow, int nbl, int64_t* seg) {
  for (int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x; i < nrow; i += int64_t(gridDim.x) * blockDim.x) {
    const uint32_t k = keys[i];
    if (k >= uint32_t(nbl)) continue;
    if (i == 0 || keys[i - 1] != k) seg[2 * k] = i;
    if (i == nrow - 1 || keys[i + 1] != k) seg[2 * k + 1] = i + 1;
  }
}

// Channel cuts of one time block: blocks [cut_j, cut_{j+1}) of the (block number, band) changes.
// MODE 1: the block number of channel c is that of the np.int32(np.linspace(0, NChan, NChBlocks))
// boundaries with NChBlocks the length of np.arange(0, NChan, nchb) plus the trailing NChan.
// MODE 2: block number c // size with size = ceil(NChan / ceil(NChan / m)).
struct ChanCuts {
  int32_t nblk;     // MODE 1: number of linspace boundaries; MODE 2: channel block size
  double lin_step;  // MODE 1: NChan / (nblk - 1)
};

__device__ inline ChanCuts chan_cuts_mode1(double nchb, int nchan) {
#pragma clang fp contract(off)
  ChanCuts cc;
  const double step = nchb < 1.0 ? 1.0 : nchb;  // np.max([NChanBlockMax, 1])
  // len(np.arange(0, NChan, step)) = ceil(NChan / step); element i = i * step
  const double n = ceil(double(nchan) / step);
  int64_t len = int64_t(n);
  if (len < 0) len = 0;
  bool has_nchan = false;
  if (len > 0) has_nchan = (double(len - 1) * step == double(nchan));
  cc.nblk = int32_t(len + (has_nchan ? 0 : 1));
  cc.lin_step = cc.nblk > 1 ? double(nchan) / double(cc.nblk - 1) : 0.0;
  return cc;
}

// np.int32(np.linspace(0, nchan, nblk))[k]
__device__ inline int32_t lin_bound(const ChanCuts& cc, int k, int nchan) {
#pragma clang fp contract(off)
  if (k >= cc.nblk - 1) return nchan;
  return int32_t(double(k) * cc.lin_step);
}

// Block number of channel c.  MODE 1 is the rampe of ClassSmearMapping.py:582-587: the largest
// k <= nblk - 2 with bound_k <= c (the bounds do not decrease, so a guess from the step and a search
// around it finds the k that a scan from 0 would stop at); one boundary alone gives 0.
template <int MODE>
__device__ inline int32_t chan_block_of(const ChanCuts& cc, int c, int nchan) {
  if (MODE == 2) return c / cc.nblk;
  if (cc.nblk <= 2) return 0;
  int32_t k = int32_t(double(c) / cc.lin_step);
  k = k < 0 ? 0 : k > cc.nblk - 2 ? cc.nblk - 2 : k;
  while (k > 0 && lin_bound(cc, k, nchan) > c) --k;
  while (k + 1 < cc.nblk - 1 && lin_bound(cc, k + 1, nchan) <= c) ++k;
  return k;
}

// One time block's channel blocks, 64 channels a turn: a lane whose channel starts a block calls
// start(j, c) with the block's number.  Returns the number of blocks.
template <int MODE, typename F>
__device__ inline int32_t wave_channel_blocks(const ChanCuts& cc, int nchan, const int32_t* __restrict__ chan_map,
                                              F start) {
  const int lane = threadIdx.x & 63;
  int32_t n = 0;
  for (int base = 0; base < nchan; base += 64) {
    const int c = base + lane;
    bool first = false;
    if (c < nchan)
      first = c == 0 || chan_map[c] != chan_map[c - 1] ||
              chan_block_of<MODE>(cc, c, nchan) != chan_block_of<MODE>(cc, c - 1, nchan);
    const uint64_t m = __ballot(first);
    if (first) start(n + __popcll(m & ((uint64_t(1) << lane) - 1)), c);
    n += __popcll(m);
  }
  return n;
}

// x of lane j (the same in every lane)
__device__ inline double lane_value(double x, int j) {
  const int lo = __builtin_amdgcn_readlane(__double2loint(x), j), hi = __builtin_amdgcn_readlane(__double2hiint(x), j);
  return __hiloint2double(hi, lo);
}

// One baseline's walk by one wavefront (rows r[0..n) in row order).  The step lengths and the
// decorrelation spans of 64 rows are worked out a row a lane; only the running sum, which has to add
// them in row order, goes from row to row, with the row's two values broadcast from their lane.
// WRITE: descriptors at desc + blk0, record words counted from word0; otherwise only the totals.
// (A thread a baseline, each row two dependent loads, a square root and two divisions after the one
// before it, and a scan over the channels at each cut, left 32 of 1024 SIMDs busy: 2.4 ms counting
// and 2.8 ms writing for 302400 rows of 2016 baselines and 64 channels; the wavefronts take
// 131 and 149 us.)
template <int MODE, bool WRITE>
__device__ void walk_baseline(const BdaParams& P, const double* __restrict__ uvw, const uint32_t* __restrict__ r,
                              int64_t row_base, int64_t n, const int32_t* __restrict__ chan_map, int64_t* nblk_out,
                              int64_t* nwords_out, BlockDesc* __restrict__ desc, int64_t blk0, int64_t word0) {
#pragma clang fp contract(off)
  const int lane = threadIdx.x & 63;
  int64_t nblk = 0, nwords = 0;
  auto close_block = [&](int64_t t0, int64_t t1, const ChanCuts& cc) {
    const int32_t nr = int32_t(t1 - t0);
    BlockDesc* d = desc + blk0 + nblk;
    const int64_t w = word0 + nwords;
    const int32_t nc = wave_channel_blocks<MODE>(cc, P.nchan, chan_map, [&](int32_t j, int32_t c) {
      if (!WRITE) return;
      d[j].word = w + int64_t(j) * (2 + nr);
      d[j].row0 = row_base + t0;
      d[j].nrows = nr;
      d[j].ch0 = c;
      if (j > 0) d[j - 1].ch1 = c;
    });
    // both modes append the channel count as the last cut
    if (WRITE && lane == 0 && nc > 0) d[nc - 1].ch1 = P.nchan;
    nblk += nc;
    nwords += int64_t(nc) * (2 + nr);
  };
  auto cuts_of_span = [&](double span_min) {
    ChanCuts cc;
    const double m = span_min < 1.0 ? 1.0 : span_min;
    const double nb = isfinite(m) ? ceil(double(P.nchan) / m) : 1.0;
    cc.nblk = int32_t(ceil(double(P.nchan) / (nb < 1.0 ? 1.0 : nb)));
    cc.lin_step = 0.0;
    return cc;
  };
  double sum = 0.0;                               // MODE 1: |duvw| since the cut; MODE 2: phase since the first row
  double least = MODE == 1 ? 1e3 : INFINITY;      // of the block's rows: channels (1) or span (2)
  int64_t t0 = 0;
  int32_t prev = 0;
  for (int64_t base = 0; base < n; base += 64) {
    const int64_t i = base + lane;
    const int m = int(n - base < 64 ? n - base : 64);
    double step = 0.0, span = 0.0;
    if (i < n) {
      // step of row i to row i + 1, the last step repeated
      const double* x = uvw + 3 * size_t(r[i]);
      const double x0 = x[0], x1 = x[1], x2 = x[2];
      const int64_t j = (i + 1 < n) ? i : n - 2;
      double d0 = MODE == 1 ? 1e-30 : 0.0, d1 = d0, d2 = d0;  // of a baseline of one row
      if (n > 1) {
        const double* a = uvw + 3 * size_t(r[j]);
        const double* b = uvw + 3 * size_t(r[j + 1]);
        d0 = MODE == 1 ? b[0] - a[0] : a[0] - b[0];
        d1 = MODE == 1 ? b[1] - a[1] : a[1] - b[1];
        d2 = MODE == 1 ? b[2] - a[2] : a[2] - b[2];
      }
      if (MODE == 1) {
        double uv = sqrt(x0 * x0 + x1 * x1 + x2 * x2);
        uv = uv > 1e-10 ? uv : 1e-10;
        const double dnu = P.k_dnu / (uv * P.l);
        span = dnu / P.dfreq;
        step = sqrt(d0 * d0 + d1 * d1 + d2 * d2);
      } else {
        step = P.k_phase * (sqrt(d0 * d0 + d1 * d1) * P.lmax + fabs(d2) * P.nmax);
        const double ext = sqrt(x0 * x0 + x1 * x1) * P.lmax + fabs(x2) * P.nmax;
        span = (P.k_span / ext) / P.dfreq;
      }
    }
    if (MODE == 1) {
      for (int k = 0; k < m; ++k) {
        const double s = lane_value(span, k);
        if (s < least) least = s;
        sum += lane_value(step, k);
        if (sum > P.duv_cut || base + k == n - 1) {
          close_block(t0, base + k + 1, chan_cuts_mode1(least, P.nchan));
          least = 1e3;
          sum = 0.0;
          t0 = base + k + 1;
        }
      }
    } else {
      // phase-based blocks: blk_i = int32(cumsum(dph)_i / dPhi), cut where it changes
      double mine = 0.0;
      for (int k = 0; k < m; ++k) {
        sum += lane_value(step, k);
        if (lane == k) mine = sum;
      }
      const int32_t blk = int32_t(mine / P.dphi);
      int32_t before = __shfl_up(blk, 1);
      if (lane == 0) before = prev;
      uint64_t cuts = __ballot(i > 0 && i < n && (P.per_row || blk != before));
      prev = __builtin_amdgcn_readlane(blk, m - 1);
      for (int k = 0; k < m; ++k) {
        if (cuts >> k & 1) {
          close_block(t0, base + k, cuts_of_span(least));
          t0 = base + k;
          least = INFINITY;
        }
        const double s = lane_value(span, k);
        if (s < least) least = s;
      }
    }
  }
  if (MODE == 2 && n > 0) close_block(t0, n, cuts_of_span(least));
  *nblk_out = nblk;
  *nwords_out = nwords;
}

template <int MODE>
__global__ __launch_bounds__(64) void bda_count_k(BdaParams P, const double* __restrict__ uvw,
                                                  const uint32_t* __restrict__ rows, const int64_t* __restrict__ seg,
                                                  const int32_t* __restrict__ chan_map, int64_t* nblk, int64_t* nwords) {
  for (int k = int(blockIdx.x); k < P.nbl; k += int(gridDim.x)) {
    const int64_t s0 = seg[2 * k], s1 = seg[2 * k + 1];
    int64_t b = 0, w = 0;
    if (s1 > s0) walk_baseline<MODE, false>(P, uvw, rows + s0, s0, s1 - s0, chan_map, &b, &w, nullptr, 0, 0);
    if (threadIdx.x == 0) {
      nblk[k] = b;
      nwords[k] = w;
    }
  }
}

template <int MODE>
__global__ __launch_bounds__(64) void bda_walk_k(BdaParams P, const double* __restrict__ uvw,
                                                 const uint32_t* __restrict__ rows, const int64_t* __restrict__ seg,
                                                 const int32_t* __restrict__ chan_map, const int64_t* __restrict__ blk_off,
                                                 const int64_t* __restrict__ word_off, BlockDesc* __restrict__ desc) {
  for (int k = int(blockIdx.x); k < P.nbl; k += int(gridDim.x)) {
    const int64_t s0 = seg[2 * k], s1 = seg[2 * k + 1];
    int64_t b = 0, w = 0;
    if (s1 > s0)
      walk_baseline<MODE, true>(P, uvw, rows + s0, s0, s1 - s0, chan_map, &b, &w, desc, blk_off[k], word_off[k]);
  }
}

__global__ void bda_emit_k(const BlockDesc* desc, int64_t nblk, const uint32_t* rows, int32_t* out) {
  int32_t* sizes = out + 2;
  int32_t* recs = out + 2 + nblk;
  for (int64_t b = int64_t(blockIdx.x) * blockDim.x + threadIdx.x; b < nblk; b += int64_t(gridDim.x) * blockDim.x) {
    const BlockDesc d = desc[b];
    sizes[b] = 2 + d.nrows;
    int32_t* rec = recs + d.word;
    rec[0] = d.ch0;
    rec[1] = d.ch1;
    for (int32_t j = 0; j < d.nrows; ++j) rec[2 + j] = int32_t(rows[d.row0 + j]);
  }
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    out[0] = int32_t(uint32_t(uint64_t(nblk) & 0xFFFFFFFFu));
    out[1] = int32_t(nblk >> 32);
  }
}

unsigned grid_for(int64_t n, int per = 256) {
  int64_t b = (n + per - 1) / per;
  if (b > 65536) b = 65536;
  if (b < 1) b = 1;
  return unsigned(b);
}

}  // namespace

struct ddf_bda_builder {
  BdaParams P{};
  hipStream_t st = nullptr;
  int64_t nrow = 0, nblk = 0, nwords = 0;
  const double* uvw = nullptr;
  const int32_t* chan_map = nullptr;
  ddf::PoolArena arena;
  uint32_t* rows = nullptr;   // sorted rows
  int64_t* seg = nullptr;
  int64_t* blk_off = nullptr;
  int64_t* word_off = nullptr;
  ~ddf_bda_builder() { arena.close(); }
  template <typename T>
  T* alloc(size_t n) {
    return static_cast<T*>(arena.get(std::max<size_t>(n, 1) * sizeof(T), st));
  }
};

#define BDA_TRY(x)                                                                              \
  do {                                                                                          \
    hipError_t e_ = (x);                                                                        \
    if (e_ != hipSuccess) {                                                                     \
      delete B;                                                                                 \
      return bfail(DDF_EHIP, std::string(#x) + ": " + hipGetErrorString(e_));               \
    }                                                                                           \
  } while (0)

extern "C" int ddf_bda_build_create(const ddf_bda_spec* spec, const double* uvw, const int32_t* a0, const int32_t* a1,
                                    int64_t nrow, const int32_t* chan_map, const int32_t* rank, ddf_bda_builder** out,
                                    int64_t* nwords, void* stream) {
  if (!spec || !out || !nwords || (nrow > 0 && (!uvw || !a0 || !a1)) || !chan_map || !rank)
    return bfail(DDF_EINVAL, "null argument");
  if (spec->mode != 1 && spec->mode != 2) return bfail(DDF_EINVAL, "BDA mode must be 1 or 2");
  if (spec->nchan <= 0 || spec->na <= 0 || nrow < 0 || nrow >= (int64_t(1) << 32))
    return bfail(DDF_EINVAL, "bad sizes");
  ddf_bda_builder* B = new ddf_bda_builder();
  hipStream_t st = static_cast<hipStream_t>(stream);
  B->st = st;
  B->nrow = nrow;
  B->uvw = uvw;
  B->chan_map = chan_map;
  const int na = spec->na;
  const int nbl = na * (na - 1);
  BdaParams& P = B->P;
  P.mode = spec->mode;
  P.nchan = spec->nchan;
  P.nbl = nbl;
  P.duv_cut = spec->duv_cut;
  P.k_dnu = spec->k_dnu;
  P.l = spec->l;
  P.dfreq = spec->dfreq;
  P.k_phase = spec->k_phase;
  P.lmax = spec->lmax;
  P.nmax = spec->nmax;
  P.k_span = spec->k_span;
  P.dphi = spec->dphi;
  P.per_row = spec->per_row;
  uint32_t* keys = B->alloc<uint32_t>(size_t(nrow));
  uint32_t* keys2 = B->alloc<uint32_t>(size_t(nrow));
  uint32_t* rows = B->alloc<uint32_t>(size_t(nrow));
  uint32_t* rows2 = B->alloc<uint32_t>(size_t(nrow));
  int32_t* d_rank = B->alloc<int32_t>(size_t(na) * na);
  B->seg = B->alloc<int64_t>(2 * size_t(nbl));
  int64_t* cnt = B->alloc<int64_t>(2 * size_t(nbl) + 2);
  B->blk_off = B->alloc<int64_t>(size_t(nbl) + 1);
  B->word_off = B->alloc<int64_t>(size_t(nbl) + 1);
  if (!keys || !keys2 || !rows || !rows2 || !d_rank || !B->seg || !cnt || !B->blk_off || !B->word_off) {
    delete B;
    return bfail(DDF_ENOMEM, "BDA builder allocation failed");
  }
  BDA_TRY(hipMemcpyAsync(d_rank, rank, size_t(na) * na * sizeof(int32_t), hipMemcpyHostToDevice, st));
  if (nrow > 0) {
    hipLaunchKernelGGL(bda_keys_k, dim3(grid_for(nrow)), dim3(256), 0, st, a0, a1, nrow, d_rank, na, nbl, keys, rows);
    BDA_TRY(hipGetLastError());
    int end_bit = 1;
    while ((int64_t(1) << end_bit) <= nbl) ++end_bit;
    hipcub::DoubleBuffer<uint32_t> dk(keys, keys2), dv(rows, rows2);
    size_t tmp_bytes = 0;
    BDA_TRY(hipcub::DeviceRadixSort::SortPairs(nullptr, tmp_bytes, dk, dv, int(nrow), 0, end_bit, st));
    void* tmp = B->alloc<char>(tmp_bytes);
    if (!tmp) {
      delete B;
      return bfail(DDF_ENOMEM, "BDA sort workspace allocation failed");
    }
    BDA_TRY(hipcub::DeviceRadixSort::SortPairs(tmp, tmp_bytes, dk, dv, int(nrow), 0, end_bit, st));
    keys = dk.Current();
    B->rows = dv.Current();
  } else {
    B->rows = rows;
  }
  hipLaunchKernelGGL(bda_fill64_k, dim3(grid_for(2 * int64_t(nbl))), dim3(256), 0, st, B->seg, 2 * int64_t(nbl),
                     int64_t(0));
  if (nrow > 0)
    hipLaunchKernelGGL(bda_segments_k, dim3(grid_for(nrow)), dim3(256), 0, st, keys, nrow, nbl, B->seg);
  int64_t* nb = cnt;
  int64_t* nw = cnt + nbl + 1;
  if (P.mode == 1)
    hipLaunchKernelGGL(bda_count_k<1>, dim3(grid_for(nbl, 1)), dim3(64), 0, st, P, uvw, B->rows, B->seg, chan_map, nb, nw);
  else
    hipLaunchKernelGGL(bda_count_k<2>, dim3(grid_for(nbl, 1)), dim3(64), 0, st, P, uvw, B->rows, B->seg, chan_map, nb, nw);
  BDA_TRY(hipGetLastError());
  hipLaunchKernelGGL(bda_fill64_k, dim3(1), dim3(64), 0, st, nb + nbl, int64_t(1), int64_t(0));
  hipLaunchKernelGGL(bda_fill64_k, dim3(1), dim3(64), 0, st, nw + nbl, int64_t(1), int64_t(0));
  size_t scan_bytes = 0;
  BDA_TRY(hipcub::DeviceScan::ExclusiveSum(nullptr, scan_bytes, nb, B->blk_off, nbl + 1, st));
  void* stmp = B->alloc<char>(scan_bytes);
  if (!stmp) {
    delete B;
    return bfail(DDF_ENOMEM, "BDA scan workspace allocation failed");
  }
  BDA_TRY(hipcub::DeviceScan::ExclusiveSum(stmp, scan_bytes, nb, B->blk_off, nbl + 1, st));
  BDA_TRY(hipcub::DeviceScan::ExclusiveSum(stmp, scan_bytes, nw, B->word_off, nbl + 1, st));
  int64_t tot[2] = {0, 0};
  BDA_TRY(hipMemcpyAsync(&tot[0], B->blk_off + nbl, sizeof(int64_t), hipMemcpyDeviceToHost, st));
  BDA_TRY(hipMemcpyAsync(&tot[1], B->word_off + nbl, sizeof(int64_t), hipMemcpyDeviceToHost, st));
  BDA_TRY(hipStreamSynchronize(st));
  B->nblk = tot[0];
  B->nwords = 2 + tot[0] + tot[1];
  *nwords = B->nwords;
  *out = B;
  return DDF_OK;
}

extern "C" int ddf_bda_build_write(ddf_bda_builder* B, int32_t* out, int64_t n, void* stream) {
  if (!B || !out) return bfail(DDF_EINVAL, "null argument");
  if (n < B->nwords) return bfail(DDF_EINVAL, "output shorter than the map");
  hipStream_t st = static_cast<hipStream_t>(stream);
  BlockDesc* desc = nullptr;
  hipError_t ea = ddf::pool_alloc(reinterpret_cast<void**>(&desc), size_t(B->nblk ? B->nblk : 1) * sizeof(BlockDesc), st);
  if (ea != hipSuccess) return bfail(DDF_EHIP, std::string("BDA descriptors: ") + hipGetErrorString(ea));
  const BdaParams& P = B->P;
  if (P.mode == 1)
    hipLaunchKernelGGL(bda_walk_k<1>, dim3(grid_for(P.nbl, 1)), dim3(64), 0, st, P, B->uvw, B->rows, B->seg,
                       B->chan_map, B->blk_off, B->word_off, desc);
  else
    hipLaunchKernelGGL(bda_walk_k<2>, dim3(grid_for(P.nbl, 1)), dim3(64), 0, st, P, B->uvw, B->rows, B->seg,
                       B->chan_map, B->blk_off, B->word_off, desc);
  hipError_t e = hipGetLastError();
  if (e == hipSuccess) {
    hipLaunchKernelGGL(bda_emit_k, dim3(grid_for(B->nblk)), dim3(256), 0, st, desc, B->nblk, B->rows, out);
    e = hipGetLastError();
  }
  (void)hipFreeAsync(desc, st);
  if (e != hipSuccess) return bfail(DDF_EHIP, std::string("BDA map kernels: ") + hipGetErrorString(e));
  return DDF_OK;
}

extern "C" int ddf_bda_build_destroy(ddf_bda_builder* B) {
  delete B;
  return DDF_OK;
}
