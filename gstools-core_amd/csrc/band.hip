// Band-limited evaluation of fields on structured grids.
//
// The modes with |kap_d| <= K_d on every axis d (kap = k / 2 pi) make up a
// band-limited function, which its values on a coarse uniform grid determine:
// with the Kaiser-Bessel window phi of kBandWidth nodes and the node spacing
// h_d = 1 / (2 kBandSigma K_d) (kBandSigma times the Nyquist rate),
//   e^{2 pi i kap x} = (1 / phihat(kap h)) sum_i phi((x - x_i) / h) e^{2 pi i kap x_i}
// to about 5e-8 (the aliases of kap beyond 1/h, window width 10 and sigma 1.5;
// Kaiser's window, J. D. Jackson et al., IEEE Trans. Med. Imaging 10, 1991,
// use it the same way).  So the band's part of the field is evaluated on the
// nodes, with amplitudes divided by phihat on every axis, and interpolated
// to the grid axis by axis, kBandWidth multiply-adds per value and axis.
// A smooth field on a fine mesh (256^3, l = 16: 39^3 nodes) costs a few
// hundredths of its modes-times-points sum this way.
//
// The modes outside the band (the far tail of a heavy-tailed spectrum,
// non-finite ones) keep the factored GEMM, run before band_finish adds the
// band's part.  k_band_plan chooses K on the device, from the axes' extents
// and the modes, by a cost model of both parts; where nothing is gained the
// band is empty and the GEMM does everything.
//
//   k_band_plan     the band, its nodes, the two mode lists
//   k_band_tables   e^{2 pi i kap x_i} per axis, node and mode (FP64); window
//                   weights per grid coordinate (FP64)
//   k_band_nodes    node values on the FP64 matrix cores, the modes split
//                   over blocks where the nodes are few
//   k_band_last     the last axis (FP64: it sums the splits and is small)
//   k_band_mid      3-D: the middle axis (FP32)
//   k_band_first    the first axis (FP32), into the output
// An axis with no more coordinates than it would need nodes keeps its
// coordinates as nodes (ident: the interpolation along it is a copy).
#include "gsc_band.h"
#include "gsc_device.h"

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>

namespace gsc {
namespace {

constexpr int kBandWidth = 10;
constexpr int kWeightLd = 12;  // floats per coordinate in the weight tables of axes 0 and 1
constexpr double kBandSigma = 1.5;
constexpr double kPi = 3.14159265358979323846264338327950288;
constexpr double kBeta = kPi * kBandWidth * (1.0 - 1.0 / (2.0 * kBandSigma));

typedef double f64x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

// Window: I0(beta sqrt(1 - (2 u / W)^2)) / c0 over |u| <= W / 2, c0 = W
// sinh(beta) / beta, so that phihat(0) = 1.
__device__ __forceinline__ double window(double u, double c0) {
  const double t = 2.0 * u / kBandWidth;
  return cyl_bessel_i0(kBeta * sqrt(fmax(0.0, 1.0 - t * t))) / c0;
}
// phihat(f) = int phi(u) e^{-2 pi i f u} du, |f| <= 1 / (2 sigma).
__device__ __forceinline__ double window_hat(double f) {
  const double a = kPi * kBandWidth * f;
  const double z = sqrt(kBeta * kBeta - a * a);
  return (sinh(z) / z) * (kBeta / sinh(kBeta));
}

// ---- the plan ----------------------------------------------------------------
constexpr int kPlanThreads = 1024;
constexpr int kQuantBins = 256;  // quarter octaves of |kap_d|
constexpr int kBandBins = 512;   // sixteenth octaves of max_d |kap_d| / q_d
constexpr int kNodeTile = 64;    // rows and columns of a node-value tile
constexpr int kNodeModes = 16;   // modes per chunk of the node sums

// Seconds of the parts, for the plan: measured on one MI355X (256 CUs).
constexpr double kCus = 256.0;
constexpr double kGemmChunk = 1.45e-6;  // a 32-mode double chunk half of a 256 x 128 GEMM tile
constexpr double kNodeChunk = 1.2e-6;   // a 16-mode chunk of a 64 x 64 node tile, one CU
constexpr double kNodeFixed = 30e-6;    // the path's own launches
constexpr double kNodeFixedShared = 5e-7;
constexpr double kStreamByte = 1.0 / 3.5e12;  // intermediate arrays, read or written

__device__ __forceinline__ int axis_nodes(double ext, double kmax) {
  // nodes of an axis of extent ext for |kap| <= kmax; a huge count saturates
  const double v = ceil(ext * kmax * (2.0 * kBandSigma)) + (kBandWidth + 1);
  return v < 1e6 ? static_cast<int>(v) : 1000000;
}

__device__ double gemm_seconds(const BandReal& R, int m) {
  if (m <= 0) return 0.0;
  const double tiles = static_cast<double>(R.gemm_tiles);
  const double rounds = R.shared ? tiles / kCus : ceil(tiles / kCus);
  return rounds * (2 * ((m + 31) / 32)) * kGemmChunk + (R.shared ? 0.0 : 5e-6);
}

__device__ double band_seconds(const BandReal& R, const int (&n)[3], int n_in, int n_rest) {
  const double rows = static_cast<double>(n[0]) * n[1], cols = static_cast<double>(n[2]) * R.ncomp;
  const double tiles = ceil(rows / kNodeTile) * ceil(cols / kNodeTile);
  const double chunks = (n_in + kNodeModes - 1) / kNodeModes;
  const double node = tiles * chunks * kNodeChunk / kCus;
  const double N1 = static_cast<double>(R.len[1]), N2 = static_cast<double>(R.len[2]);
  const double c = R.ncomp;
  const double stream = 4.0 * c * (2.0 * rows * N2 + (R.dim == 3 ? 2.0 * n[0] * N1 * N2 : 0.0));
  const double outb = 4.0 * c * R.len[0] * N1 * N2 * (n_rest > 0 ? 3.0 : 1.0);
  return node + (stream + outb) * kStreamByte + (R.shared ? kNodeFixedShared : kNodeFixed) +
         gemm_seconds(R, n_rest);
}

__device__ __forceinline__ void block_minmax(double& lo, double& hi, double (*red)[2]) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) {
    lo = fmin(lo, __shfl_xor(lo, off, 64));
    hi = fmax(hi, __shfl_xor(hi, off, 64));
  }
  __syncthreads();
  if ((threadIdx.x & 63) == 0) {
    red[threadIdx.x >> 6][0] = lo;
    red[threadIdx.x >> 6][1] = hi;
  }
  __syncthreads();
#pragma unroll
  for (int w = 0; w < kPlanThreads / 64; ++w) {
    lo = fmin(lo, red[w][0]);
    hi = fmax(hi, red[w][1]);
  }
}

// Axis d of kap: a 2-D grid's second axis sits in place 2.
__device__ __forceinline__ int kap_axis(int dim, int d) { return dim == 2 && d == 2 ? 1 : d; }

__global__ void __launch_bounds__(kPlanThreads)
k_band_plan(BandReal* __restrict__ dr, BandState* __restrict__ st, const BandReal one,
            bool use_one) {
  __shared__ int qh[3][kQuantBins];
  __shared__ int hist[kBandBins];
  __shared__ double red[kPlanThreads / 64][2];
  __shared__ double s_q[3];
  __shared__ int wcnt[kPlanThreads / 64];
  __shared__ double wcost[kPlanThreads / 64];
  __shared__ int wbin[kPlanThreads / 64];
  __shared__ BandState S;
  // one grid: its description comes as an argument and is left in dr[0] for
  // the kernels after this one
  const BandReal R = use_one ? one : dr[blockIdx.x];
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
  if (use_one && tid == 0) dr[0] = one;
  const int M = R.M, dim = R.dim;
  for (int i = tid; i < 3 * kQuantBins; i += kPlanThreads) (&qh[0][0])[i] = 0;
  for (int i = tid; i < kBandBins; i += kPlanThreads) hist[i] = 0;
  // extents of the finite coordinates
  double ext[3], lo[3];
#pragma unroll
  for (int d = 0; d < 3; ++d) {
    double a = INFINITY, b = -INFINITY;
    if (!(dim == 2 && d == 1))
      for (int64_t i = tid; i < R.len[d]; i += kPlanThreads) {
        const double x = R.ax[d][i];
        if (isfinite(x)) {
          a = fmin(a, x);
          b = fmax(b, x);
        }
      }
    block_minmax(a, b, red);
    lo[d] = a <= b ? a : 0.0;
    ext[d] = a <= b ? b - a : 0.0;
  }
  __syncthreads();
  // q_d: 0.9 quantile of |kap_d| (to a quarter octave), the band's shape
  for (int m = tid; m < M; m += kPlanThreads) {
    const ModeRec r = R.modes[m];
#pragma unroll
    for (int d = 0; d < 3; ++d) {
      if (dim == 2 && d == 1) continue;
      const double k = fabs(r.kap[kap_axis(dim, d)]);
      const int b = k > 0.0 ? static_cast<int>(fmin(fmax(floor(4.0 * log2(k)) + kQuantBins / 2, 0.0),
                                                    kQuantBins - 1.0))
                            : 0;
      if (isfinite(k)) atomicAdd(&qh[d][b], 1);
    }
  }
  __syncthreads();
  if (wv < 3) {  // wave d scans histogram d, four bins per lane
    int c[4], sum = 0;
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      c[u] = qh[wv][4 * lane + u];
      sum += c[u];
    }
    int inc = sum;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const int y = __shfl_up(inc, o, 64);
      if (lane >= o) inc += y;
    }
    const int total = __shfl(inc, 63, 64);
    const int want = (9 * total + 9) / 10;
    int run = inc - sum;
    if (total == 0 && lane == 0) s_q[wv] = 1.0;
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      if (run < want && want <= run + c[u])
        s_q[wv] = exp2((4 * lane + u + 1 - kQuantBins / 2) / 4.0);
      run += c[u];
    }
  }
  __syncthreads();
  // bin of a mode: sixteenth octaves of its largest |kap_d| / q_d; the last
  // bin is never in the band (non-finite modes, values far out)
  auto bin_of = [&](const ModeRec& r) {
    double s = 0.0;
    bool ok = isfinite(r.th);
#pragma unroll
    for (int d = 0; d < 3; ++d) {
      if (dim == 2 && d == 1) continue;
      const double k = fabs(r.kap[kap_axis(dim, d)]);
      ok = ok && isfinite(k);
      s = fmax(s, k / s_q[d]);
    }
    ok = ok && isfinite(r.amp[0]);
    // the incompressible projector is 0 / 0 for k = 0: left to the GEMM
    if (R.ncomp > 1 && s == 0.0) ok = false;
    if (!ok) return kBandBins - 1;
    if (!(s > 0.0)) return 0;
    return static_cast<int>(
        fmin(fmax(floor(16.0 * log2(s)) + kBandBins / 2, 0.0), kBandBins - 1.0));
  };
  for (int m = tid; m < M; m += kPlanThreads) atomicAdd(&hist[bin_of(R.modes[m])], 1);
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
  double cost = INFINITY;
  if (tid < kBandBins - 1 && cnt > 0) {
    const double edge = exp2((tid + 1 - kBandBins / 2) / 16.0);
    int n[3];
    bool fits = true;
#pragma unroll
    for (int d = 0; d < 3; ++d) {
      n[d] = dim == 2 && d == 1 ? 1 : axis_nodes(ext[d], edge * s_q[d]);
      if (n[d] >= R.len[d]) n[d] = static_cast<int>(R.len[d]);
      fits = fits && n[d] <= R.cap[d];
    }
    const double nodes = static_cast<double>(n[0]) * n[1] * n[2] * R.ncomp;
    if (fits && nodes <= static_cast<double>(R.fcap)) cost = band_seconds(R, n, inc, M - inc);
  }
  int best = tid;
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    const double c2 = __shfl_xor(cost, o, 64);
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
  int top = cost < gemm_seconds(R, M) ? best : -1;  // bins 0 .. top are in
  // the largest |kap_d| of the band gives the spacing
  double km[3] = {0.0, 0.0, 0.0};
  if (top >= 0)
    for (int m = tid; m < M; m += kPlanThreads) {
      const ModeRec r = R.modes[m];
      if (bin_of(r) <= top)
#pragma unroll
        for (int d = 0; d < 3; ++d)
          if (!(dim == 2 && d == 1)) km[d] = fmax(km[d], fabs(r.kap[kap_axis(dim, d)]));
    }
#pragma unroll
  for (int d = 0; d < 3; ++d) {
    double z = 0.0;
    block_minmax(z, km[d], red);
  }
  int n[3], ident[3];
  double h[3], x0[3];
#pragma unroll
  for (int d = 0; d < 3; ++d) {
    n[d] = 1;
    ident[d] = 1;
    h[d] = 1.0;
    x0[d] = 0.0;
    if (dim == 2 && d == 1) continue;
    n[d] = min(axis_nodes(ext[d], km[d]), R.cap[d] < R.len[d] ? R.cap[d] : 1000000);
    if (n[d] >= R.len[d]) {
      n[d] = static_cast<int>(R.len[d]);
      continue;
    }
    ident[d] = 0;
    // the coarsest spacing the band allows; any for a constant axis
    h[d] = km[d] > 0.0 ? 1.0 / (2.0 * kBandSigma * km[d]) : (ext[d] > 0.0 ? ext[d] : 1.0);
    if (h[d] > ext[d] && ext[d] > 0.0) h[d] = ext[d];
    x0[d] = lo[d] - 0.5 * kBandWidth * h[d];
  }
  const int64_t nodes = static_cast<int64_t>(n[0]) * n[1] * n[2] * R.ncomp;
  // (the choice above counted at least these nodes; never past the workspace)
  if (nodes > R.fcap || n[0] > R.cap[0] || n[1] > R.cap[1] || n[2] > R.cap[2]) top = -1;
  // mode lists, both in order: the band's with their deconvolved amplitude
  // (and the output scale), the rest as they are
  int ns = 0, nr = 0;
  for (int base = 0; base < M; base += kPlanThreads) {
    const int m = base + tid;
    ModeRec r{};
    bool in = false;
    if (m < M) {
      r = R.modes[m];
      in = top >= 0 && bin_of(r) <= top;
    }
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
        double a = static_cast<double>(r.amp[0]) * R.scale;
#pragma unroll
        for (int d = 0; d < 3; ++d)
          if (!ident[d]) a /= window_hat(r.kap[kap_axis(dim, d)] * h[d]);
        double* q = R.bm + 5 * static_cast<int64_t>(ns + before);
        q[0] = r.kap[0];
        q[1] = dim == 2 ? 0.0 : r.kap[1];
        q[2] = r.kap[dim == 2 ? 1 : 2];
        q[3] = r.th;
        q[4] = a;
      } else {
        R.rest[nr + (tid - before)] = r;
      }
    }
    ns += total;
    nr += min(kPlanThreads, M - base) - total;
  }
  if (tid == 0) {
    S.n_in = ns;
    S.n_rest = nr;
#pragma unroll
    for (int d = 0; d < 3; ++d) {
      S.n[d] = n[d];
      S.ident[d] = ident[d];
      S.lo[d] = x0[d];
      S.h[d] = h[d];
    }
    // splits of the modes: enough node-tile items to fill the chip, at least
    // four chunks of modes each, the partial sums within F
    const int64_t tiles = ((static_cast<int64_t>(n[0]) * n[1] + kNodeTile - 1) / kNodeTile) *
                          ((static_cast<int64_t>(n[2]) * R.ncomp + kNodeTile - 1) / kNodeTile);
    int64_t sp = (R.shared ? 4 : 1024) / tiles;
    sp = min(sp, static_cast<int64_t>(ns) / (4 * kNodeModes));
    sp = min(sp, R.fcap / (nodes > 0 ? nodes : 1));
    S.splits = static_cast<int>(max(sp, static_cast<int64_t>(1)));
    st[blockIdx.x] = S;
  }
}

// ---- tables ----------------------------------------------------------------
// Modes of the tables are padded to whole chunks with zeros in the first
// axis' table (the others' pads repeat the last mode and meet those zeros).
__device__ __forceinline__ int pad_modes(int n) {
  return (n + kNodeModes - 1) / kNodeModes * kNodeModes;
}

__global__ void __launch_bounds__(256)
k_band_tables(const BandReal* __restrict__ dr, const BandState* __restrict__ st) {
  const BandReal& R = dr[blockIdx.y];
  const BandState S = st[blockIdx.y];
  if (S.n_in == 0) return;
  const int dim = R.dim;
  const int mp = pad_modes(S.n_in);
  const int64_t step = static_cast<int64_t>(gridDim.x) * 256;
  const int64_t t0 = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
  for (int d = 0; d < 3; ++d) {
    if (dim == 2 && d == 1) continue;
    const int cols = S.n[d] * (d == 2 ? R.ncomp : 1);
    const int ld = R.cap[d] * (d == 2 ? R.ncomp : 1);
    double2* tab = R.tab[d];
    for (int64_t e = t0; e < static_cast<int64_t>(mp) * cols; e += step) {
      const int m = static_cast<int>(e / cols), col = static_cast<int>(e - static_cast<int64_t>(m) * cols);
      const int comp = col / S.n[d], node = col - comp * S.n[d];
      const double* q = R.bm + 5 * static_cast<int64_t>(min(m, S.n_in - 1));
      const double x = S.ident[d] ? R.ax[d][node] : S.lo[d] + node * S.h[d];
      double t = q[d] * x;
      if (d == 0) t += q[3];
      double sn, cs;
      sincospi(2.0 * (t - rint(t)), &sn, &cs);
      double a = d == 0 ? (m < S.n_in ? q[4] : 0.0) : 1.0;
      if (d == 2 && R.ncomp > 1) {
        // projector delta_c0 - k_c k_0 / |k|^2 (field.rs:138-151)
        const double kc = comp == 0 ? q[0] : (dim == 2 || comp == 2 ? q[2] : q[1]);
        a = (comp == 0 ? 1.0 : 0.0) - kc * q[0] / (q[0] * q[0] + q[1] * q[1] + q[2] * q[2]);
      }
      tab[static_cast<int64_t>(m) * ld + col] = make_double2(a * cs, a * sn);
    }
  }
  // window weights of the grid's coordinates; a non-finite one gets NaN
  const double c0 = kBandWidth * sinh(kBeta) / kBeta;
  for (int d = 0; d < 3; ++d) {
    if (S.ident[d]) continue;
    const int64_t len = R.len[d];
    for (int64_t e = t0; e < len * kBandWidth; e += step) {
      const int k = static_cast<int>(e / len);
      const int64_t i = e - k * len;
      const double x = R.ax[d][i];
      int f = 0;
      double w = NAN;
      if (isfinite(x)) {
        const double u = (x - S.lo[d]) / S.h[d];
        f = min(max(static_cast<int>(ceil(u - 0.5 * kBandWidth)), 0), S.n[d] - kBandWidth);
        w = window(u - (f + k), c0);
      }
      if (d == 2) R.wt2[e] = w;
      else R.wt[d][i * kWeightLd + k] = static_cast<float>(w);
      if (k == 0) R.i0[d][i] = f;
    }
  }
}

// ---- node values ------------------------------------------------------------
// F[row][col] = sum_m Im(P(row, m) C(m, col)), row = (i, j) over the first
// two axes, P = tab0[m][i] tab1[m][j], C = tab2: a real product over K = 2
// modes, (Re P, Im P) against (Im C, Re C), on v_mfma_f64_16x16x4f64 (lane
// layouts as in krige.hip).  A block of four waves takes 64 x 64 tiles (32 x
// 32 per wave) and one split of the modes; 16 modes per chunk go through
// LDS, the next chunk's table values are loaded during the MFMAs.
constexpr int kNodeLd = kNodeTile + 16;  // LDS row: the four k rows of a read on two bank halves
__global__ void __launch_bounds__(256)
k_band_nodes(const BandReal* __restrict__ dr, const BandState* __restrict__ st) {
  __shared__ double sa[2 * kNodeModes][kNodeLd];
  __shared__ double sb[2 * kNodeModes][kNodeLd];
  const BandReal& R = dr[blockIdx.y];
  const BandState S = st[blockIdx.y];
  if (S.n_in == 0) return;
  const int n1 = S.n[1];
  const int rows = S.n[0] * n1, cols = S.n[2] * R.ncomp;
  const int rt = (rows + kNodeTile - 1) / kNodeTile, ct = (cols + kNodeTile - 1) / kNodeTile;
  const int chunks = pad_modes(S.n_in) / kNodeModes;
  const bool two = R.dim == 3;
  const auto g0 = global_ptr(R.tab[0]), g1 = global_ptr(R.tab[1]), g2 = global_ptr(R.tab[2]);
  const int64_t ld0 = R.cap[0], ld1 = R.cap[1], ld2 = static_cast<int64_t>(R.cap[2]) * R.ncomp;
  const int lane = threadIdx.x & 63, g = lane >> 4, jl = lane & 15;
  const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wr = 32 * (wv >> 1), wc = 32 * (wv & 1);
  const int64_t items = static_cast<int64_t>(rt) * ct * S.splits;
  for (int64_t it = blockIdx.x; it < items; it += gridDim.x) {
    const int sp = static_cast<int>(it % S.splits);
    const int64_t tile = it / S.splits;
    const int r0 = static_cast<int>(tile / ct) * kNodeTile;
    const int c0 = static_cast<int>(tile % ct) * kNodeTile;
    const int q0 = static_cast<int>(static_cast<int64_t>(chunks) * sp / S.splits);
    const int q1 = static_cast<int>(static_cast<int64_t>(chunks) * (sp + 1) / S.splits);
    // this thread's table columns: row r0 + lane and column c0 + lane
    // (clamped: rows and columns past the end are not stored)
    const int row = min(r0 + lane, rows - 1), col = min(c0 + lane, cols - 1);
    const int ri = row / n1, rj = row - ri * n1;
    double2 p0[4], p1[4], p2[4];
    auto gload = [&](int q) {
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const int64_t m = q * kNodeModes + wv + 4 * u;
        p0[u].x = g0[m * ld0 + ri].x;
        p0[u].y = g0[m * ld0 + ri].y;
        if (two) {
          p1[u].x = g1[m * ld1 + rj].x;
          p1[u].y = g1[m * ld1 + rj].y;
        }
        p2[u].x = g2[m * ld2 + col].x;
        p2[u].y = g2[m * ld2 + col].y;
      }
    };
    f64x4 acc[2][2];
#pragma unroll
    for (int a = 0; a < 2; ++a)
#pragma unroll
      for (int b = 0; b < 2; ++b) acc[a][b] = f64x4{0.0, 0.0, 0.0, 0.0};
    if (q0 < q1) gload(q0);
    for (int q = q0; q < q1; ++q) {
      __syncthreads();  // the previous chunk is read
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const int k = 2 * (wv + 4 * u);
        double re = p0[u].x, im = p0[u].y;
        if (two) {
          re = p0[u].x * p1[u].x - p0[u].y * p1[u].y;
          im = p0[u].x * p1[u].y + p0[u].y * p1[u].x;
        }
        sa[k][lane] = re;
        sa[k + 1][lane] = im;
        sb[k][lane] = p2[u].y;
        sb[k + 1][lane] = p2[u].x;
      }
      __syncthreads();
      if (q + 1 < q1) gload(q + 1);
#pragma unroll
      for (int kk = 0; kk < 2 * kNodeModes; kk += 4) {
        double a[2], b[2];
#pragma unroll
        for (int t = 0; t < 2; ++t) {
          a[t] = sa[kk + g][wr + 16 * t + jl];
          b[t] = sb[kk + g][wc + 16 * t + jl];
        }
#pragma unroll
        for (int x = 0; x < 2; ++x)
#pragma unroll
          for (int y = 0; y < 2; ++y)
            acc[x][y] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[x], b[y], acc[x][y], 0, 0, 0);
      }
    }
    double* F = R.F + static_cast<int64_t>(sp) * rows * cols;
#pragma unroll
    for (int x = 0; x < 2; ++x)
#pragma unroll
      for (int y = 0; y < 2; ++y)
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          const int r = r0 + wr + 16 * x + 4 * v + g, c = c0 + wc + 16 * y + jl;
          if (r < rows && c < cols) F[static_cast<int64_t>(r) * cols + c] = acc[x][y][v];
        }
  }
}

// ---- interpolation ------------------------------------------------------------
// Last axis: t1[comp][row][c] from the nodes of row (FP64 sums, splits added
// in order); a block takes one (row, comp) at a time.
constexpr int kLineMax = 2048;  // nodes of a line held in LDS
__global__ void __launch_bounds__(256)
k_band_last(const BandReal* __restrict__ dr, const BandState* __restrict__ st) {
  __shared__ double line[kLineMax];
  const BandReal& R = dr[blockIdx.y];
  const BandState S = st[blockIdx.y];
  if (S.n_in == 0) return;
  const int rows = S.n[0] * S.n[1], n2 = S.n[2], cols = n2 * R.ncomp;
  const int64_t len = R.len[2], fs = static_cast<int64_t>(rows) * cols;
  const auto wt = global_ptr(R.wt2);
  const auto i0 = global_ptr(R.i0[2]);
  const auto F = global_ptr(R.F);
  const auto t1 = global_ptr(R.t1);
  for (int64_t it = blockIdx.x; it < static_cast<int64_t>(rows) * R.ncomp; it += gridDim.x) {
    const int comp = static_cast<int>(it / rows);
    const int64_t row = it - static_cast<int64_t>(comp) * rows;
    __syncthreads();  // the previous line is read
    for (int k = threadIdx.x; k < n2; k += 256) {
      const int64_t e = row * cols + comp * n2 + k;
      double v = 0.0;
      for (int s = 0; s < S.splits; ++s) v += F[s * fs + e];
      line[k] = v;
    }
    __syncthreads();
    for (int64_t c = threadIdx.x; c < len; c += 256) {
      double v = 0.0;
      if (S.ident[2]) {
        v = line[c];
      } else {
        const int f = i0[c];
#pragma unroll
        for (int k = 0; k < kBandWidth; ++k) v = __builtin_fma(wt[k * len + c], line[f + k], v);
      }
      t1[it * len + c] = static_cast<float>(v);
    }
  }
}

// One axis in FP32: out[p][q] (p over the axis' coordinates) from in[node][q],
// q over `width` values, kVec per lane; a lane keeps the window of nodes in
// registers while p walks over a run of coordinates and reads nodes only when
// the window moves.  ADD: out += (the factored GEMM's part is there).
template <int V> struct VecT;
template <> struct VecT<1> { using type = float; };
template <> struct VecT<4> { using type = f32x4; };

// Constant-memory view of a pointer to what an earlier kernel wrote: uniform
// reads through it are scalar loads.
template <typename T>
__device__ __forceinline__ const __attribute__((address_space(4))) T* const_ptr(const T* p) {
  return (const __attribute__((address_space(4))) T*)(p);  // address-space conversion
}

template <int V, bool ADD, typename InP, typename OutP>
__device__ __forceinline__ void band_run(InP in, OutP out, const float* weights,
                                         const int* first, int64_t len, int64_t width, int ident,
                                         int64_t q, int64_t p0, int64_t p1) {
  const auto wt = const_ptr(weights);
  const auto i0 = const_ptr(first);
  using T = typename VecT<V>::type;
  T win[kBandWidth];
  int cur = -(1 << 30);
  for (int64_t p = p0; p < p1; ++p) {
    T v;
    if (ident) {
      v = *reinterpret_cast<const __attribute__((address_space(1))) T*>(in + p * width + q);
    } else {
      const int f = i0[p];
      if (f != cur) {
        if (f == cur + 1) {
#pragma unroll
          for (int k = 0; k + 1 < kBandWidth; ++k) win[k] = win[k + 1];
          win[kBandWidth - 1] = *reinterpret_cast<const __attribute__((address_space(1))) T*>(
              in + static_cast<int64_t>(f + kBandWidth - 1) * width + q);
        } else {
#pragma unroll
          for (int k = 0; k < kBandWidth; ++k)
            win[k] = *reinterpret_cast<const __attribute__((address_space(1))) T*>(
                in + static_cast<int64_t>(f + k) * width + q);
        }
        cur = f;
      }
      const auto wp = wt + p * kWeightLd;
      v = win[0] * wp[0];
#pragma unroll
      for (int k = 1; k < kBandWidth; ++k) {
        const float w = wp[k];
        if constexpr (V == 1) {
          v = __builtin_fmaf(win[k], w, v);
        } else {
#pragma unroll
          for (int c = 0; c < V; ++c) v[c] = __builtin_fmaf(win[k][c], w, v[c]);
        }
      }
    }
    auto* o = reinterpret_cast<__attribute__((address_space(1))) T*>(out + p * width + q);
    if constexpr (ADD) *o = *o + v;
    else __builtin_nontemporal_store(v, o);
  }
}

// Middle axis of a 3-D grid: t2[comp][i][b][c] from t1[comp][i][j][c].
constexpr int kMidRun = 32;
__global__ void __launch_bounds__(256)
k_band_mid(const BandReal* __restrict__ dr, const BandState* __restrict__ st) {
  const BandReal& R = dr[blockIdx.y];
  const BandState S = st[blockIdx.y];
  if (S.n_in == 0 || R.dim != 3) return;
  const int64_t len = R.len[1], width = R.len[2];
  const int64_t qb = (width + 255) / 256, pb = (len + kMidRun - 1) / kMidRun;
  const int64_t planes = static_cast<int64_t>(S.n[0]) * R.ncomp;
  for (int64_t it = blockIdx.x; it < planes * qb * pb; it += gridDim.x) {
    const int64_t plane = it / (qb * pb), r = it - plane * (qb * pb);
    const int64_t q = (r % qb) * 256 + threadIdx.x, p0 = r / qb * kMidRun;
    if (q < width)
      band_run<1, false>(global_ptr(R.t1) + plane * S.n[1] * width,
                                 global_ptr(R.t2) + plane * len * width, R.wt[1], R.i0[1], len, width, S.ident[1], q, p0,
                                 min(p0 + kMidRun, len));
  }
}

// First axis, into the output.
constexpr int kFirstRun = 32;
template <int V>
__device__ __forceinline__ void band_first(const BandReal& R, const BandState& S) {
  const int64_t len = R.len[0], width = R.len[1] * R.len[2];
  const int64_t qb = (width + 256 * V - 1) / (256 * V), pb = (len + kFirstRun - 1) / kFirstRun;
  const float* src = R.dim == 3 ? R.t2 : R.t1;
  for (int64_t it = blockIdx.x; it < R.ncomp * qb * pb; it += gridDim.x) {
    const int64_t comp = it / (qb * pb), r = it - comp * (qb * pb);
    const int64_t q = ((r % qb) * 256 + threadIdx.x) * V, p0 = r / qb * kFirstRun;
    if (q >= width) continue;
    const auto in = global_ptr(src) + comp * S.n[0] * width;
    const auto out = global_ptr(R.out) + comp * len * width;
    const int64_t p1 = min(p0 + kFirstRun, len);
    if (S.n_rest > 0)
      band_run<V, true>(in, out, R.wt[0], R.i0[0], len, width, S.ident[0],
                        q, p0, p1);
    else
      band_run<V, false>(in, out, R.wt[0], R.i0[0], len, width, S.ident[0],
                         q, p0, p1);
  }
}
__global__ void __launch_bounds__(256)
k_band_first(const BandReal* __restrict__ dr, const BandState* __restrict__ st) {
  const BandReal& R = dr[blockIdx.y];
  const BandState S = st[blockIdx.y];
  if (S.n_in == 0) return;
  // four values per lane where every row of the output keeps 16-byte
  // alignment (the workspace arrays do, their rows being as long)
  const bool vec = R.len[1] * R.len[2] % 4 == 0 &&
                   (reinterpret_cast<uintptr_t>(R.out) & 15) == 0;
  if (vec) band_first<4>(R, S);
  else band_first<1>(R, S);
}

}  // namespace

BandPlan plan_band(int dim, int64_t M, const int64_t* shape, int ncomp) {
  BandPlan p{};
  p.ncomp = ncomp;
  p.len[0] = shape[0];
  p.len[1] = dim == 3 ? shape[1] : 1;
  p.len[2] = shape[dim - 1];
  const int64_t N = p.len[0] * p.len[1] * p.len[2];
  if (dim < 2 || M <= 0 || N <= 0) return p;
  constexpr int64_t kT2Max = int64_t(1) << 28;  // values of t2: 1 GiB
  for (int d = 0; d < 3; ++d) {
    // at most half as many nodes as coordinates, or all of a short axis
    const int64_t c = std::min<int64_t>(p.len[d], p.len[d] / 2 + kBandWidth + 2);
    p.cap[d] = static_cast<int>(std::min<int64_t>(c, d == 2 ? kLineMax : 1 << 20));
  }
  if (dim == 3) {
    const int64_t plane = p.len[1] * p.len[2] * ncomp;
    p.cap[0] = static_cast<int>(std::min<int64_t>(p.cap[0], kT2Max / plane));
  }
  // FP64 node sums cost about six times the GEMM's per value
  p.fcap = std::max<int64_t>(N * ncomp / 6, 1 << 16);
  const int64_t rows = static_cast<int64_t>(p.cap[0]) * p.cap[1];
  const int64_t t1max = std::min<int64_t>(rows, p.fcap) * p.len[2] * ncomp;
  p.on = p.cap[0] > 0 && p.fcap < (int64_t(1) << 31) && t1max < (int64_t(1) << 29);
  if (!p.on) return p;
  size_t off = 0;
  auto take = [&off](size_t b) {
    const size_t o = off;
    off += (b + 255) & ~static_cast<size_t>(255);
    return o;
  };
  const size_t mp = static_cast<size_t>(M + kNodeModes);
  p.rest = take(sizeof(ModeRec) * static_cast<size_t>(M));
  p.bm = take(sizeof(double) * 5 * static_cast<size_t>(M));
  for (int d = 0; d < 3; ++d) {
    if (dim == 2 && d == 1) continue;
    p.tab[d] = take(sizeof(double2) * mp * static_cast<size_t>(p.cap[d]) * (d == 2 ? ncomp : 1));
    p.i0[d] = take(sizeof(int) * static_cast<size_t>(p.len[d]));
    p.wt[d] = take((d == 2 ? sizeof(double) * kBandWidth : sizeof(float) * kWeightLd) *
                   static_cast<size_t>(p.len[d]));
  }
  p.F = take(sizeof(double) * static_cast<size_t>(p.fcap));
  p.t1 = take(sizeof(float) * static_cast<size_t>(t1max));
  if (dim == 3)
    p.t2 = take(sizeof(float) * static_cast<size_t>(p.cap[0]) * p.len[1] * p.len[2] * ncomp);
  p.bytes = off;
  return p;
}

void band_place(const BandPlan& p, void* base, BandReal* r) {
  char* b = static_cast<char*>(base);
  r->ncomp = p.ncomp;
  r->fcap = p.fcap;
  r->rest = reinterpret_cast<ModeRec*>(b + p.rest);
  r->bm = reinterpret_cast<double*>(b + p.bm);
  for (int d = 0; d < 3; ++d) {
    r->len[d] = p.len[d];
    r->cap[d] = p.cap[d];
    r->tab[d] = reinterpret_cast<double2*>(b + p.tab[d]);
    r->i0[d] = reinterpret_cast<int*>(b + p.i0[d]);
    r->wt[d] = reinterpret_cast<float*>(b + p.wt[d]);
  }
  r->wt2 = reinterpret_cast<double*>(b + p.wt[2]);
  r->F = reinterpret_cast<double*>(b + p.F);
  r->t1 = reinterpret_cast<float*>(b + p.t1);
  r->t2 = reinterpret_cast<float*>(b + p.t2);
}

namespace {
// Blocks per grid: one grid takes the chip, an ensemble's share it.
unsigned blocks_x(int count, int64_t want) {
  return static_cast<unsigned>(std::max<int64_t>(1, std::min<int64_t>(want, 16384 / count + 1)));
}
}  // namespace

hipError_t launch_band_plan(BandReal* d, BandState* st, int count, const BandReal* one,
                            hipStream_t s) {
  k_band_plan<<<count, kPlanThreads, 0, s>>>(d, st, one ? *one : BandReal{}, one != nullptr);
  k_band_tables<<<dim3(blocks_x(count, 1024), count), 256, 0, s>>>(d, st);
  k_band_nodes<<<dim3(blocks_x(count, 1024), count), 256, 0, s>>>(d, st);
  return hipGetLastError();
}

hipError_t launch_band_finish(const BandReal* d, BandState* st, int count, int64_t max_out,
                              hipStream_t s) {
  k_band_last<<<dim3(blocks_x(count, 2048), count), 256, 0, s>>>(d, st);
  k_band_mid<<<dim3(blocks_x(count, 4096), count), 256, 0, s>>>(d, st);
  const int64_t want = std::min<int64_t>(4096, (max_out / (256 * kFirstRun) + 1) * 2);
  k_band_first<<<dim3(blocks_x(count, want), count), 256, 0, s>>>(d, st);
  return hipGetLastError();
}

}  // namespace gsc
