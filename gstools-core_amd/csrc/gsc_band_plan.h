// The plan of the band-limited paths (band.hip: grids, band_points.hip: point
// lists), one block of kPlanThreads threads: which modes are in the band, its
// nodes, and the two mode lists.
#pragma once

#include "gsc_band.h"
#include "gsc_device.h"
#include "gsc_local.h"

#include <hip/hip_runtime.h>

namespace gsc {
namespace {

constexpr int kBandWidth = 8;
constexpr double kBandSigma = 2.0;
constexpr double kPi = 3.14159265358979323846264338327950288;
constexpr double kBeta = kPi * kBandWidth * (1.0 - 1.0 / (2.0 * kBandSigma));

// 1 / phihat(f), phihat(f) = int phi(u) e^{-2 pi i f u} du = (sinh(z) / z)
// (beta / sinh(beta)), z^2 = beta^2 - (pi W f)^2: a Chebyshev fit of degree 9
// in (2 sigma f)^2 over the band |f| <= 1 / (2 sigma), to 1.1e-11.
template <typename T>
__device__ __forceinline__ T window_hat_inv(T f) {
  static_assert(kBandWidth == 8 && kBandSigma == 2.0, "the fit is for this window");
  constexpr double c[10] = {0.9999999999891889,    0.9916419977861659,   0.5176792547568738,
                            0.18969587705046465,   0.05487719688349006,  0.013390516468031443,
                            0.0028095623888406774, 0.0006117128781691989, 4.809348127997348e-05,
                            3.6267606186861704e-05};
  const T v = static_cast<T>(2.0 * kBandSigma) * f * (static_cast<T>(2.0 * kBandSigma) * f);
  T r = static_cast<T>(c[9]);
#pragma unroll
  for (int i = 8; i >= 0; --i) r = r * v + static_cast<T>(c[i]);
  return r;
}

// ---- the plan ----------------------------------------------------------------
constexpr int kPlanThreads = 512;
constexpr int kAxisWaves = 2;    // waves that read one axis; three axes
static_assert(3 * kAxisWaves <= kPlanThreads / 64, "waves for every axis");
constexpr int kLastRows = 16;    // node lines per work item of k_band_last, at most
constexpr int kMidRun = 16;      // coordinates per run of k_band_mid
constexpr int kFirstRun = 16;    // and of k_band_first, one grid
constexpr int kBandBins = 512;   // sixteenth octaves of max_d |kap_d| / q_d
static_assert(kBandBins <= kPlanThreads, "a thread per bin");
constexpr int kNodeModes = 16;   // modes per chunk of the node sums

// Seconds of the parts, for the plan: measured on one MI355X (256 CUs).
// FP32: the plan runs on one CU, and its choices are coarse.
constexpr float kCus = 256.0f;
constexpr float kNodeChunk64 = 0.50e-6f;   // a 16-mode chunk of a 64 x 64 node tile, one CU
constexpr float kNodeChunk128 = 1.05e-6f;  // of a 128 x 128 one
constexpr float kNodeChunkAlone = 0.8e-6f;  // of a 64 x 64 one alone on its CU
constexpr float kNodeFixed = 30e-6f;    // the path's own launches
constexpr float kStreamByte = 1.0f / 5e12f;  // arrays read or written (first axis: 5 to 6 TB/s)

__device__ __forceinline__ float axis_nodes(double ext, double kmax) {
  // nodes of an axis of extent ext for |kap| <= kmax; a huge count saturates
  const double v = ceil(ext * kmax * (2.0 * kBandSigma)) + (kBandWidth + 1);
  return v < 1e6 ? static_cast<float>(v) : 1e6f;
}

__device__ float gemm_seconds(const BandReal& R, int m) {
  return factored_seconds(R.gemm_tiles, m, R.shared != 0);
}

// Seconds of a chunk over all node tiles; big: 128 x 128 tiles, where they
// are less work and, for one grid, enough to fill the chip.
__host__ __device__ __forceinline__ float node_tiles(float rows, float cols, bool shared, bool& big) {
  const float t1 = ceilf(rows / 64) * ceilf(cols / 64) * kNodeChunk64;
  const float n2 = ceilf(rows / 128) * ceilf(cols / 128);
  big = n2 * kNodeChunk128 < t1 && (shared || n2 >= kCus);
  return big ? n2 * kNodeChunk128 : t1;
}

// Splits of n_in modes over the blocks of a node tile: enough items to fill the
// chip, at least two chunks of modes each, the partial sums within F.
__device__ __forceinline__ int node_splits(const BandReal& R, float rows, float cols, bool big,
                                           int n_in) {
  const float tb = big ? 128.0f : 64.0f;
  const float tiles = ceilf(rows / tb) * ceilf(cols / tb);
  float sp = (R.shared ? 4.0f : 768.0f) / tiles;
  sp = fminf(sp, static_cast<float>(n_in / (2 * kNodeModes)));
  // (a little below the exact quotient: floats)
  sp = fminf(sp, 0.9999f * static_cast<float>(R.fcap) / fmaxf(rows * cols, 1.0f));
  return max(static_cast<int>(sp), 1);
}

__device__ float band_seconds(const BandReal& R, const float (&n)[3], int n_in, int n_rest) {
  const float rows = n[0] * n[1], cols = n[2] * R.ncomp;
  bool big;
  float chunk = node_tiles(rows, cols, R.shared, big) / kCus;
  // one grid: an item's chunks run one after the other, and F may have no room for
  // splits (197 x 699 x 2 values of 1396 modes: 28 items of 82 us)
  if (!R.shared && !big)
    chunk = fmaxf(chunk, kNodeChunkAlone / node_splits(R, rows, cols, big, n_in));
  const float node = chunk * ((n_in + kNodeModes - 1) / kNodeModes);
  const float N1 = static_cast<float>(R.len[1]), N2 = static_cast<float>(R.len[2]);
  const float stream = 2.0f * rows * N2 + (R.dim == 3 ? 2.0f * n[0] * N1 * N2 : 0.0f);
  const float outb = static_cast<float>(R.len[0]) * N1 * N2 * (n_rest > 0 ? 3.0f : 1.0f);
  return node + (stream + outb) * (4.0f * kStreamByte) * R.ncomp +
         (R.shared ? 0.0f : kNodeFixed) + gemm_seconds(R, n_rest);
}

// Point lists (3-D).  A wave interpolates 64 points of a cell from a window of
// 2 tiles x 16 x 16 nodes (tiles of the matrix product), so the cells are at
// most (2 tiles - W, 16 - W, 15 - W) nodes wide, less a margin for rounding (the
// last axis' window starts at an even node).  Few tiles per window are less
// work, many allow wider and so fewer cells: the fewest that keep within the
// cells there may be.
constexpr int kWinTiles[3] = {5, 6, 8};
constexpr float kWinWork[3] = {1.0f, 1.2f, 1.6f}, kWinWorkVec[3] = {1.0f, 1.7f, 2.2f};
constexpr int kWinCols = 16;
constexpr double kWinMargin = 0.1;
__device__ __forceinline__ int window_nodes(int d, int tiles) {
  return d == 0 ? 2 * tiles : (d == 1 ? kWinCols : kWinCols - 1);
}
// Modes right at the band's edge alias to 7e-7 of themselves, and the nodes'
// FP32 and fp16 roundings are noise of 1e-7 of the root of the deconvolved
// amplitudes' power: the nodes are kPointEdge closer than the band needs, or
// kPointEdgeWide where the deconvolved amplitudes have more than kPointNoise
// times the field's power (the modes of a k-grid, many of them near the faces),
// which keeps the error below the local kernel's.  Grids are kPointEdge closer
// for the Fourier method (256^3, 1000 modes, l = 16: 3.3e-7 at 1, 1.4e-7 at 1.1,
// the factored GEMM 3.4e-7).  Against 64 bits, sigma = 1: 1000 modes of a k-grid
// at 2e6 points, l = 20: 3.1e-7 at 1, 1.3e-7 here, the local kernel 2.8e-7; 700
// Gaussian ones at 1e6 points, l = 5: 1.8e-7 at 1, 1.6e-7 here, the local kernel
// 2.3e-7.
constexpr double kPointEdge = 1.1, kPointEdgeWide = 1.18;
constexpr float kPointNoise = 4.0f;
constexpr float kPointLocal = 1.0e-13f;     // a point-mode of the local kernel
constexpr float kPointLocalVec = 1.75e-13f;
constexpr float kPointRough = 6e-13f;       // its point-mode of a rough mode
constexpr float kPointRest = 2.7e-13f;      // of the FP64-phase loop over the rest modes
constexpr float kPointWin = 2.5e-11f;       // a point of the interpolation
constexpr float kPointWinVec = 2.9e-11f;    // a point and component of it, and of the results' way back
constexpr float kPointCells = 30e-6f;       // the sort over as many cells as there may be
constexpr float kPointFixed = 12e-6f;       // the path's own launches
constexpr double kPointCell = 4096.0;       // target points per cell

// Fewer points leave most of the chip idle, and a mode costs its latency at least:
// a rest mode (four points per lane) 0.26 to 0.29 us whatever the points, a rough
// mode of the local kernel (one point per lane, many waves) a third of that, the node
// sums a chunk of all modes in turn where F has no room for splits.  Slopes over the
// mode count at 1e5 to 3e5 points; without them 200000 points of 2000 exponential
// modes took the band, 169 us in a box of 150 and 284 in one of 500 (l = 20), for the
// local kernel's 131 and 165.  The band has to be clearly ahead there: latencies that
// are not counted make up more of both.
constexpr int64_t kPointFew = 300000;
constexpr float kPointSure = 0.6f;
constexpr float kFewLocalMode = 2.4e-8f;  // a smooth mode: its cells' part
constexpr float kFewRough = 2.2e-13f, kFewRoughVec = 2.8e-13f;  // a slot of a rough mode,
constexpr float kFewRoughMore = 1.0e-13f, kFewRoughMoreVec = 6e-13f;  // and of those past
constexpr float kFewRoughMany = 400.0f;   // as many, whose list leaves the scalar caches
constexpr float kFewRoughMode = 0.065e-6f, kFewRoughModeVec = 0.17e-6f;  // at least
constexpr float kFewRestMode = 0.29e-6f, kFewRestModeVec = 0.26e-6f;     // at least
constexpr float kFewSumWord = 1e-12f;     // a node value read or written by the sum of the splits

// The local kernel with n_rough modes beyond its widest phase at the smallest cells.
__device__ __forceinline__ float points_seconds_off(const PointsArgs& A, int M, int n_rough) {
  float slots = static_cast<float>(A.N), s = 0.0f;
  const bool most = n_rough > 0.005f * M;  // as many cells as there may be
  if (most) slots += A.all_cells * (0.5f * kWavePts);
  const float local = A.vec ? kPointLocalVec : kPointLocal;
  if (A.N < kPointFew) {
    const float smooth = fmaxf(slots * local, A.N * local + kFewLocalMode);
    const float rough = slots * (n_rough * (A.vec ? kFewRoughVec : kFewRough) +
                                 fmaxf(n_rough - kFewRoughMany, 0.0f) *
                                     (A.vec ? kFewRoughMoreVec : kFewRoughMore));
    return kPointSure * ((M - n_rough) * smooth +
                         fmaxf(rough, n_rough * (A.vec ? kFewRoughModeVec : kFewRoughMode)));
  }
  if (most) s = kPointCells;
  return s + slots * ((M - n_rough) * local + n_rough * kPointRough);
}
__device__ __forceinline__ float points_seconds(const BandReal& R, const PointsArgs& A,
                                                const float (&n)[3], int n_in, int n_rest) {
  const float rows = n[0] * n[1], cols = n[2] * R.ncomp;
  bool big;
  float chunk = node_tiles(rows, cols, false, big) / kCus;
  float rest = A.N * kPointRest, sum = 0.0f;
  if (A.N < kPointFew) {
    const int sp = node_splits(R, rows, cols, big, n_in);
    if (!big) chunk = fmaxf(chunk, kNodeChunkAlone / sp);
    sum = rows * cols * ((sp + 1) * kFewSumWord);
    rest = fmaxf(rest, A.vec ? kFewRestModeVec : kFewRestMode);
  }
  const float node = chunk * ((n_in + kNodeModes - 1) / kNodeModes) + sum;
  const float N = static_cast<float>(A.N);
  // cells at each window, as cell_grid counts them
  auto along = [](float nodes, int win) {
    const float c = fmaxf(ceilf((nodes - (kBandWidth + 1)) /
                                (win - kBandWidth - static_cast<float>(kWinMargin))), 1.0f);
    const float f = ceilf(c * 0.125f);
    return f * ceilf(c / f);
  };
  const float c12 = along(n[1], window_nodes(1, 0)) * along(n[2], window_nodes(2, 0));
  float work = INFINITY, cells = 0.0f;
#pragma unroll
  for (int v = 2; v >= 0; --v) {
    const float c = c12 * along(n[0], window_nodes(0, kWinTiles[v]));
    if (c <= static_cast<float>(A.max_cells)) {
      work = A.vec ? kWinWorkVec[v] : kWinWork[v];
      cells = c;
    }
  }
  // (cells of few points leave slots of their waves empty)
  const float slots = N + cells * (0.5f * kWavePts);
  return node + slots * work * (A.vec ? kPointWinVec * R.ncomp : kPointWin) +
         rest * n_rest + kPointFixed;
}
// Cells of an axis of extent ext with nodes h apart.
__device__ __forceinline__ int window_cells(double ext, double h, int win) {
  const double v = ceil(ext / (h * (win - kBandWidth - kWinMargin)));
  return static_cast<int>(fmin(fmax(v, 1.0), 1e6));
}

// Largest (MAX) or sum of v[i] over the block's threads, in every thread.
template <int K, bool MAX>
__device__ __forceinline__ void block_reduce(float (&v)[K], float (*red)[4]) {
  auto op = [](float a, float b) { return MAX ? fmaxf(a, b) : a + b; };
#pragma unroll
  for (int off = 32; off > 0; off >>= 1)
#pragma unroll
    for (int i = 0; i < K; ++i) v[i] = op(v[i], __shfl_xor(v[i], off, 64));
  __syncthreads();
  if ((threadIdx.x & 63) == 0)
#pragma unroll
    for (int i = 0; i < K; ++i) red[threadIdx.x >> 6][i] = v[i];
  __syncthreads();
  const int l = threadIdx.x & (kPlanThreads / 64 - 1);
#pragma unroll
  for (int i = 0; i < K; ++i) {
    v[i] = red[l][i];
#pragma unroll
    for (int off = kPlanThreads / 128; off > 0; off >>= 1) v[i] = op(v[i], __shfl_xor(v[i], off, 64));
  }
}

struct PlanWave {  // |kap| per axis place
  float x, y, z;
  int ok;          // finite, as the amplitudes
  float amp;       // largest |amplitude|, where ok
  __device__ __forceinline__ float at(int d) const { return d == 0 ? x : (d == 1 ? y : z); }
};

// By a block of kPlanThreads threads.  R in registers or constant memory.
template <bool POINTS>
__device__ __forceinline__ void band_plan(const BandReal& R, const PointsArgs& A,
                                          BandState* __restrict__ st, int* __restrict__ any_rest) {
  __shared__ int hist[kBandBins];
  __shared__ float red[kPlanThreads / 64][4];
  __shared__ double wax[kPlanThreads / 64][POINTS ? 6 : 2];
  __shared__ int wcnt[kPlanThreads / 64];
  __shared__ float wcost[kPlanThreads / 64];
  __shared__ int wbin[kPlanThreads / 64];
  __shared__ BandState S;
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
  const int M = R.M, dim = R.dim;
  double margin = POINTS || R.k_grid ? kPointEdge : 1.0 + 0x1p-22;  // of the nodes over the band
  // the thread's modes are tid, tid + kPlanThreads, ..; the wave numbers of the
  // first two stay in registers: |kap| per axis place, and whether it is finite
  auto read = [&](const ModeRec& r) {
    // (amplitudes the window's factors, and the points' sum of them, do not take to
    // infinity)
    constexpr float most = POINTS ? 0x1p96f : 0x1p120f;
    bool ok = isfinite(r.th) && fabsf(r.amp[0]) < most;
    if constexpr (POINTS) ok = ok && fabsf(r.amp[1]) < most && fabsf(r.amp[2]) < most;
    // (a 2-D grid's second axis sits in place 2)
    const float x = fabsf(static_cast<float>(r.kap[0])), y = fabsf(static_cast<float>(r.kap[1])),
                z = fabsf(static_cast<float>(r.kap[2]));
    PlanWave k{x, dim == 2 ? 0.0f : y, dim == 2 ? y : z, 0, 0.0f};
    k.ok = ok && isfinite(k.x) && isfinite(k.y) && isfinite(k.z);
    if constexpr (POINTS)
      if (k.ok) k.amp = fmaxf(fabsf(r.amp[0]), fmaxf(fabsf(r.amp[1]), fabsf(r.amp[2])));
    return k;
  };
  PlanWave ka{}, kb{};
  const ModeRec first = load_mode(R.modes, min(tid, M - 1));  // for the lists
  if (tid < M) ka = read(first);
  if (tid + kPlanThreads < M) kb = read(load_mode(R.modes, tid + kPlanThreads));
  auto waves = [&](int m) {
    if (m >= 2 * kPlanThreads) return read(load_mode(R.modes, m));
    const bool a = m < kPlanThreads;
    return PlanWave{a ? ka.x : kb.x, a ? ka.y : kb.y, a ? ka.z : kb.z, a ? ka.ok : kb.ok,
                    a ? ka.amp : kb.amp};
  };
  for (int i = tid; i < kBandBins; i += kPlanThreads) hist[i] = 0;
  // extents of the finite coordinates: the largest x and -x
  if constexpr (POINTS) {
    double a[6];
#pragma unroll
    for (int c = 0; c < 6; ++c) a[c] = -INFINITY;
    for (int i = tid; i < kBoxBlocks; i += kPlanThreads)
#pragma unroll
      for (int d = 0; d < 3; ++d) {
        a[2 * d] = fmax(a[2 * d], A.box[i * 6 + 2 * d + 1]);
        a[2 * d + 1] = fmax(a[2 * d + 1], -A.box[i * 6 + 2 * d]);
      }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1)
#pragma unroll
      for (int c = 0; c < 6; ++c) a[c] = fmax(a[c], __shfl_xor(a[c], off, 64));
    if (lane == 0)
#pragma unroll
      for (int c = 0; c < 6; ++c) wax[wv][c] = a[c];
  } else {  // kAxisWaves waves per axis
    double a = -INFINITY, b = -INFINITY;
    const int d = wv / kAxisWaves;
    if (d < 3 && !(dim == 2 && d == 1)) {  // uniform per wave
      const double* ax = d == 0 ? R.ax[0] : (d == 1 ? R.ax[1] : R.ax[2]);
      const int64_t len = d == 0 ? R.len[0] : (d == 1 ? R.len[1] : R.len[2]);
      for (int64_t i = (wv - d * kAxisWaves) * 64 + lane; i < len; i += 64 * kAxisWaves) {
        const double x = ax[i];
        if (isfinite(x)) {
          a = fmax(a, x);
          b = fmax(b, -x);
        }
      }
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
      a = fmax(a, __shfl_xor(a, off, 64));
      b = fmax(b, __shfl_xor(b, off, 64));
    }
    if (lane == 0) {
      wax[wv][0] = a;
      wax[wv][1] = b;
    }
  }
  // q_d, the geometric mean of |kap_d|: the shape of the band, which a heavy
  // tail does not stretch; and the largest |kap_d| of all, which bounds every axis,
  // and amplitude
  float ls[4] = {0.0f, 0.0f, 0.0f, 0.0f}, kall[4] = {0.0f, 0.0f, 0.0f, 0.0f};
  int cnt0[3] = {0, 0, 0};
  for (int m = tid; m < M; m += kPlanThreads) {
    const PlanWave k = waves(m);
    kall[3] = fmaxf(kall[3], k.amp);
#pragma unroll
    for (int d = 0; d < 3; ++d) {
      if (isfinite(k.at(d))) kall[d] = fmaxf(kall[d], k.at(d));
      const float l = __log2f(k.at(d));
      if (isfinite(l)) {
        ls[d] += l;
        ++cnt0[d];
      }
    }
  }
  block_reduce<4, true>(kall, red);
  // (the counts, up to M, in one float: only a mean's scale hangs on them)
  ls[3] = static_cast<float>(max(cnt0[0], max(cnt0[1], cnt0[2])));
  block_reduce<4, false>(ls, red);
  float s_q[3];
#pragma unroll
  for (int d = 0; d < 3; ++d) s_q[d] = exp2f(ls[d] / fmaxf(ls[3], 1.0f));
  double ext[3], lo[3];
#pragma unroll
  for (int d = 0; d < 3; ++d) {  // (block_reduce synchronised the block)
    double a = -INFINITY, b = -INFINITY;
    if constexpr (POINTS) {
#pragma unroll
      for (int w = 0; w < kPlanThreads / 64; ++w) {
        a = fmax(a, wax[w][2 * d]);
        b = fmax(b, wax[w][2 * d + 1]);
      }
    } else {
#pragma unroll
      for (int w = 0; w < kAxisWaves; ++w) {
        a = fmax(a, wax[d * kAxisWaves + w][0]);
        b = fmax(b, wax[d * kAxisWaves + w][1]);
      }
    }
    const bool any = a >= -b;
    lo[d] = any ? -b : 0.0;
    ext[d] = any ? a + b : 0.0;
  }
  // bin of a mode: sixteenth octaves of its largest |kap_d| / q_d; the last
  // bin is never in the band (non-finite modes, values far out)
  auto bin_of = [&](const PlanWave& k) {
    bool ok = k.ok;
    float s = 0.0f;
#pragma unroll
    for (int d = 0; d < 3; ++d)
      if (!(dim == 2 && d == 1)) s = fmaxf(s, k.at(d) / s_q[d]);
    // the incompressible projector is 0 / 0 for k = 0: left to the GEMM
    if (R.ncomp > 1 && !(s > 0.0f)) ok = false;
    if (!ok) return kBandBins - 1;
    return static_cast<int>(fminf(fmaxf(floorf(16.0f * __log2f(s)) + kBandBins / 2, 0.0f),
                                  kBandBins - 1.0f));
  };
  float rough[1] = {0.0f};
  if constexpr (POINTS) {
    // the local kernel's rough modes at its smallest cells (near-cubic ones
    // over the axes with an extent)
    float vol = 1.0f, active = 0.0f;
#pragma unroll
    for (int d = 0; d < 3; ++d)
      if (ext[d] > 0.0) {
        vol *= static_cast<float>(ext[d]);
        active += 1.0f;
      }
    const float hh = active > 0.0f
                         ? 0.5f * exp2f(__log2f(vol / A.all_cells) / active)
                         : 0.0f;
    for (int m = tid; m < M; m += kPlanThreads) {
      const PlanWave k = waves(m);
      float sum = 0.0f;
#pragma unroll
      for (int d = 0; d < 3; ++d)
        if (ext[d] > 0.0) sum += k.at(d);
      if (!(sum * hh <= 1.0f)) rough[0] += 1.0f;
    }
    block_reduce<1, false>(rough, red);
  }
  for (int m = tid; m < M; m += kPlanThreads) {
    atomicAdd(&hist[bin_of(waves(m))], 1);
  }
  __syncthreads();
  // thread b: cost with the modes of the bins up to b in the band
  const int cnt = tid < kBandBins ? hist[tid] : 0;
  int inc = cnt;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const int y = __shfl_up(inc, o, 64);
    if (lane >= o) inc += y;
  }
  if (lane == 63) wcnt[wv] = inc;
  __syncthreads();
  for (int w = 0; w < wv; ++w) inc += wcnt[w];
  float cost = INFINITY;
  if (tid < kBandBins - 1 && cnt > 0) {
    const float edge = exp2f((tid + 1 - kBandBins / 2) / 16.0f);
    float n[3];
    bool fits = true;
#pragma unroll
    for (int d = 0; d < 3; ++d) {
      n[d] = dim == 2 && d == 1 ? 1.0f : axis_nodes(
          ext[d], fmin(static_cast<double>(edge) * s_q[d], static_cast<double>(kall[d])) * margin);
      if constexpr (POINTS) n[d] = fmaxf(n[d] + (d == 2 ? 1.0f : 0.0f), static_cast<float>(kWinCols));
      else n[d] = fminf(n[d], static_cast<float>(R.len[d]));
      fits = fits && n[d] <= R.cap[d];
    }
    if (fits && n[0] * n[1] * n[2] * R.ncomp <= static_cast<float>(R.fcap)) {
      if constexpr (POINTS) cost = points_seconds(R, A, n, inc, M - inc);
      else cost = band_seconds(R, n, inc, M - inc);
    }
  }
  int best = tid;
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    const float c2 = __shfl_xor(cost, o, 64);
    const int b2 = __shfl_xor(best, o, 64);
    if (c2 < cost || (c2 == cost && b2 < best)) {
      cost = c2;
      best = b2;
    }
  }
  if (lane == 0) {
    wcost[wv] = cost;
    wbin[wv] = best;
  }
  __syncthreads();
  cost = wcost[0];
  best = wbin[0];
#pragma unroll
  for (int w = 1; w < kPlanThreads / 64; ++w)
    if (wcost[w] < cost) {
      cost = wcost[w];
      best = wbin[w];
    }
  float off_cost;
  if constexpr (POINTS) off_cost = points_seconds_off(A, M, static_cast<int>(rough[0]));
  else off_cost = gemm_seconds(R, M);
  int top = cost < off_cost ? best : -1;  // bins 0 .. top are in
  // the largest |kap_d| of the band gives the spacing
  float kf[3] = {0.0f, 0.0f, 0.0f};
  if (top >= 0)
    for (int m = tid; m < M; m += kPlanThreads) {
      const PlanWave k = waves(m);
      if (bin_of(k) <= top)
#pragma unroll
        for (int d = 0; d < 3; ++d) kf[d] = fmaxf(kf[d], k.at(d));
    }
  block_reduce<3, true>(kf, red);
  if constexpr (POINTS)
    if (top >= 0) {  // uniform
      // noise of the node values: the deconvolved amplitudes' power (over the largest)
      float q[2] = {0.0f, 0.0f};
      int ea = 0;
      (void)frexpf(kall[3], &ea);
      for (int m = tid; m < M; m += kPlanThreads) {
        const PlanWave k = waves(m);
        float a = 0.0f;
#pragma unroll
        for (int c = 0; c < 3; ++c) {
          const float s = ldexpf(R.modes[m].amp[c], -ea);
          a += s * s;
        }
        if (!isfinite(a)) continue;
        q[1] += a;
        if (bin_of(k) > top) continue;
#pragma unroll
        for (int d = 0; d < 3; ++d) {
          const float f = kf[d] > 0.0f ? k.at(d) / (kf[d] * static_cast<float>(2.0 * kBandSigma *
                                                                              kPointEdge))
                                       : 0.0f;
          const float w = window_hat_inv(f);
          a *= w * w;
        }
        q[0] += a;
      }
      block_reduce<2, false>(q, red);
      if (q[0] > kPointNoise * q[1]) margin = kPointEdgeWide;
    }
  // (rounded up: no |kap_d| of the band is above)
  const double km[3] = {kf[0] * margin, kf[1] * margin, kf[2] * margin};
  int n[3], ident[3];
  double h[3], x0[3];
#pragma unroll
  for (int d = 0; d < 3; ++d) {
    n[d] = 1;
    ident[d] = 1;
    h[d] = 1.0;
    x0[d] = 0.0;
    if (dim == 2 && d == 1) continue;
    if constexpr (POINTS) {
      n[d] = max(static_cast<int>(axis_nodes(ext[d], km[d])), kWinCols);
      if (d == 2) n[d] += n[d] & 1;
    } else {
      n[d] = static_cast<int>(axis_nodes(ext[d], km[d]));
      if (n[d] >= R.len[d]) {
        n[d] = static_cast<int>(R.len[d]);
        continue;
      }
    }
    ident[d] = 0;
    // the coarsest spacing the band allows, within what is finite (its inverse is
    // needed too: not the extent of an axis that has next to none)
    const double most = 1024.0 * fmax(ext[d], 1.0);
    h[d] = km[d] > 0.0 ? fmin(1.0 / (2.0 * kBandSigma * km[d]), most) : most;
    x0[d] = lo[d] - 0.5 * kBandWidth * h[d];
  }
  // (a count past its bound is at most 1e6, so the product of three fits)
  const int64_t nodes = static_cast<int64_t>(n[0]) * n[1] * n[2] * R.ncomp;
  // (the choice above counted at least these nodes; never past the workspace)
  if (nodes > R.fcap || n[0] > R.cap[0] || n[1] > R.cap[1] || n[2] > R.cap[2]) top = -1;
  if constexpr (POINTS)
    // points so far out that their places in nodes, of three rounded coordinates, are
    // no longer good to window_base's 1e-6: the local kernel
#pragma unroll
    for (int d = 0; d < 3; ++d)
      if (fmax(fabs(lo[d]), fabs(lo[d] + ext[d])) > 1e9 * h[d]) top = -1;
  if constexpr (POINTS) {
    // the cells: windows' width at most, about kPointCell points at most
    __shared__ BinParams P;
    if (tid == 0) {
      double vol = 1.0;
      int active = 0;
      for (int d = 0; d < 3; ++d)
        if (ext[d] > 0.0) {
          vol *= ext[d];
          ++active;
        }
      const double side =
          active > 0 ? pow(vol / fmax(1.0, A.N / kPointCell), 1.0 / active) : 1.0;
      P.band = 0;
      for (int v = 0; v < 3 && top >= 0 && !P.band; ++v) {
        int c[3] = {1, 1, 1}, need[3];
        for (int d = 0; d < 3; ++d) {
          need[d] = ext[d] > 0.0 ? window_cells(ext[d], h[d], window_nodes(d, kWinTiles[v])) : 1;
          if (ext[d] > 0.0) c[d] = max(need[d], static_cast<int>(fmin(ceil(ext[d] / side), 1e6)));
        }
        // (made fewer where they are too many)
        cell_grid(c, lo, ext, A.max_cells, P);
        P.band = c[0] >= need[0] && c[1] >= need[1] && c[2] >= need[2] ? kWinTiles[v] : 0;
      }
      for (int d = 0; d < 3; ++d) {
        P.node0[d] = x0[d];
        P.inv_node[d] = 1.0 / h[d];
        P.nodes[d] = n[d];
      }
    }
    __syncthreads();
    if (P.band == 0) top = -1;
    if (tid == 0) *A.prm = P;
  }
  // mode lists, both in order: the band's with their deconvolved amplitude,
  // the rest as they are
  int ns = 0, nr = 0;
  float amax = 0.0f, asum = 0.0f;
  auto place = [&](int base, const ModeRec& r) {
    const int m = base + tid;
    const bool in = m < M && bin_of(waves(min(m, M - 1))) <= top;
    const unsigned long long bal = __ballot(in);
    __syncthreads();
    if (lane == 0) wcnt[wv] = __popcll(bal);
    __syncthreads();
    int before = __popcll(bal & ((1ull << lane) - 1)), total = 0;
#pragma unroll
    for (int w = 0; w < kPlanThreads / 64; ++w) {
      const int c = wcnt[w];
      if (w < wv) before += c;
      total += c;
    }
    if (m < M) {
      if (in) {
        BandMode q;
        q.kap[0] = r.kap[0];
        q.kap[1] = dim == 2 ? 0.0 : r.kap[1];
        q.kap[2] = r.kap[dim == 2 ? 1 : 2];
        q.th = r.th;
        // (point lists: the component amplitudes over their largest, which
        // goes into amp)
        double a = static_cast<double>(r.amp[0]);
        float big = 0.0f;
        if constexpr (POINTS) {
          big = fmaxf(fabsf(r.amp[0]), fmaxf(fabsf(r.amp[1]), fabsf(r.amp[2])));
          if (A.vec) a = big;
        }
#pragma unroll
        for (int d = 0; d < 3; ++d)
          if (!ident[d]) a *= window_hat_inv(q.kap[d] * h[d]);
        amax = fmaxf(amax, fabsf(static_cast<float>(a)));
        asum += fabsf(static_cast<float>(a));
        q.amp = static_cast<float>(a);
        // projector delta_c0 - k_c k_0 / |k|^2 (field.rs:138-151)
        float pr[3] = {1.0f, 0.0f, 0.0f};
        if constexpr (POINTS) {
          if (A.vec)
#pragma unroll
            for (int c = 0; c < 3; ++c) pr[c] = big > 0.0f ? r.amp[c] / big : 0.0f;
        } else if (R.ncomp > 1) {
          const double f = q.kap[0] / (q.kap[0] * q.kap[0] + q.kap[1] * q.kap[1] +
                                       q.kap[2] * q.kap[2]);
          pr[0] = static_cast<float>(1.0 - q.kap[0] * f);
          pr[1] = static_cast<float>(-q.kap[dim == 2 ? 2 : 1] * f);
          pr[2] = static_cast<float>(-q.kap[2] * f);
        }
#pragma unroll
        for (int c = 0; c < 3; ++c) q.proj[c] = pr[c];
        R.bm[ns + before] = q;
      } else {
        R.rest[nr + (tid - before)] = r;
      }
    }
    ns += total;
    nr += min(kPlanThreads, M - base) - total;
  };
  place(0, first);
  for (int base = kPlanThreads; base < M; base += kPlanThreads)
    place(base, load_mode(R.modes, min(base + tid, M - 1)));
  // whole chunks of modes: zero amplitudes past the last
  if (tid < kNodeModes) R.bm[ns + tid] = BandMode{};
  float am[1] = {amax}, as[1] = {asum};
  block_reduce<1, true>(am, red);
  if constexpr (POINTS) block_reduce<1, false>(as, red);
  if (tid == 0) {
    S.n_in = ns;
    S.n_rest = nr;
    // amplitudes are scaled to at most 2^14 in the fp16 products: the low parts of
    // smaller ones stay clear of the subnormals (to at most 1, a mode in the band's
    // corner, whose deconvolved amplitude is 20 times the others', cost them 1e-6)
    int e = 0;
    if (am[0] > 0.0f && am[0] < INFINITY) (void)frexpf(am[0], &e);
    e -= 14;
    S.amp_exp = -e;
    S.out_scale = R.scale * ldexp(1.0, e);
    if constexpr (POINTS) {
      // node values times 2^g stay below 2^15 (fp16 parts): as the sum of the
      // amplitudes does
      int g = 0;
      if (as[0] > 0.0f && as[0] < INFINITY) (void)frexpf(as[0], &g);
      S.g_scale = ldexp(1.0, 15 - (g - e));
      S.out_scale *= ldexp(1.0, g - e - 15);
    }
#pragma unroll
    for (int d = 0; d < 3; ++d) {
      S.n[d] = n[d];
      S.ident[d] = ident[d];
      S.lo[d] = x0[d];
      S.h[d] = h[d];
    }
    const float rows = static_cast<float>(n[0]) * n[1];
    const float cols = static_cast<float>(n[2]) * R.ncomp;
    bool big;
    (void)node_tiles(rows, cols, R.shared, big);
    S.big = big;
    const float tb = big ? 128.0f : 64.0f;
    const float tiles = ceilf(rows / tb) * ceilf(cols / tb);
    S.splits = node_splits(R, rows, cols, big, ns);
    S.items[0] = static_cast<int64_t>(tiles) * S.splits;
    if constexpr (POINTS) {
      if (ns == 0) S.items[0] = 0;
      *st = S;
    }
  }
  if (POINTS) return;
  if (tid == 0) {
    // work items of the kernels that follow
    const int64_t nrows = static_cast<int64_t>(n[0]) * n[1];
    const int64_t width = R.len[1] * R.len[2];
    // first axis: 1: 16-byte accesses where every row of the output keeps
    // their alignment (the workspace arrays do, their rows being as long); 2:
    // 16-byte accesses at any word, the row's last lane overlapping its
    // neighbour (same values; not where it would add twice): 607 MB of rows of
    // 545 columns take 177 us (aligned ones 124 us), 271 us column by column; 0:
    // as many columns per lane as a row has 256s, up to four
    S.vec = width % 4 == 0 && (reinterpret_cast<uintptr_t>(R.out) & 15) == 0 ? 1
            : nr == 0 && width >= 4                                          ? 2
                                                                             : 0;
    S.first_cols = S.vec ? 4 : static_cast<int>(min((width + 255) / 256, int64_t(4)));
    const int64_t fq = (width + 256 * S.first_cols - 1) / (256 * S.first_cols);
    // (one grid: shorter runs where there are few)
    const int64_t run = R.ncomp * fq * R.len[0] / 1024;
    S.first_run = R.shared ? R.shared
                           : static_cast<int>(max(min(run, int64_t(kFirstRun)), int64_t(4)));
    S.last_rows = R.shared ? max(min(R.shared / 4, kLastRows), 1)
                           : static_cast<int>(max(min(nrows * R.ncomp / 1024, int64_t(kLastRows)),
                                                  int64_t(1)));
    S.items[1] = (nrows * R.ncomp + S.last_rows - 1) / S.last_rows;
    S.items[2] = dim == 3 ? static_cast<int64_t>(n[0]) * R.ncomp * ((R.len[2] + 255) / 256) *
                                ((R.len[1] + kMidRun - 1) / kMidRun)
                          : 0;
    S.items[3] = R.ncomp * fq * ((R.len[0] + S.first_run - 1) / S.first_run);
    if (ns == 0) S.items[0] = S.items[1] = S.items[2] = S.items[3] = 0;
    if (any_rest && nr > 0) atomicAdd(any_rest, 1);
    *st = S;
  }
}


}  // namespace
}  // namespace gsc
