// Band-limited evaluation of fields on structured grids.
//
// The modes with |kap_d| <= K_d on every axis d (kap = k / 2 pi) make up a
// band-limited function, which its values on a coarse uniform grid determine:
// with the Kaiser-Bessel window phi of kBandWidth nodes and the node spacing
// h_d = 1 / (2 kBandSigma K_d) (kBandSigma times the Nyquist rate),
//   e^{2 pi i kap x} = (1 / phihat(kap h)) sum_i phi((x - x_i) / h) e^{2 pi i kap x_i}
// to about 1e-7 (the aliases of kap beyond 1/h, window width 8 and sigma 2;
// Kaiser's window, J. D. Jackson et al., IEEE Trans. Med. Imaging 10, 1991,
// use it the same way).  So the band's part of the field is evaluated on the
// nodes, with amplitudes divided by phihat on every axis, and interpolated
// to the grid axis by axis, kBandWidth multiply-adds per value and axis.
// A smooth field on a fine mesh (256^3, l = 16: about 45^3 nodes) costs a few
// hundredths of its modes-times-points sum this way.
//
// The modes outside the band (the far tail of a heavy-tailed spectrum,
// non-finite ones) keep the factored GEMM, run before band_finish adds the
// band's part.  k_band_plan chooses K on the device, from the axes' extents
// and the modes, by a cost model of both parts; where nothing is gained the
// band is empty and the GEMM does everything.
//
//   k_band_plan     the band, its nodes, the two mode lists (one block per
//                   grid; latency)
//   k_band_nodes    node values: split-precision fp16 products on the matrix
//                   cores, the modes split over blocks where the nodes are
//                   few; blocks of the same launch give the window weights per
//                   grid coordinate (FP64) and the rest modes' GEMM tables
//   k_band_last     the last axis (FP64: it sums the splits and is small)
//   k_band_mid      3-D: the middle axis (FP32)
//   k_band_first    the first axis (FP32), into the output (HBM)
// An axis with no more coordinates than it would need nodes keeps its
// coordinates as nodes (ident: the interpolation along it is a copy).
#include "gsc_band.h"
#include "gsc_band_plan.h"
#include "gsc_device.h"
#include "gsc_gemm.h"

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>

namespace gsc {
namespace {

constexpr int kWeightLd = 8;  // floats per coordinate in the weight tables of axes 0 and 1

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef _Float16 half2_t __attribute__((ext_vector_type(2)));
typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

// Window: I0(beta sqrt(1 - (2 u / W)^2)) / c0 over |u| <= W / 2, c0 = W
// sinh(beta) / beta, so that phihat(0) = 1.  Its taps at u = 3.5 - k - r, k < 4, as
// polynomials in r over |r| <= 1/2 (Chebyshev fits, to 2e-13), and at k - 3.5 - r
// with -r.  (The Bessel function itself took 40 us for the 16 k weights of a 1024 x
// 1024 grid by one block.)
__device__ constexpr double kTap[kBandWidth / 2][12] = {
    {3.7778122903787384e-05, 0.0003035836194710282, 0.0010435288280002089, 0.0020072802099016973,
     0.0023543182365240588, 0.0016824888952741747, 0.00063147272118408077, -2.589380995577047e-07,
     -0.00011425540964946486, -4.2313069293354799e-05, 2.4280444247421865e-06, 4.924827909379e-06},
    {0.007911188907602144, 0.02881556348988604, 0.043156193395416299, 0.032072683381108268,
     0.009141388972600353, -0.0032421838653121696, -0.0032529642118392823, -0.00054587579465299057,
     0.00031613141565810845, 0.00013835861269574193, -8.237036552375746e-06, -1.3410615254039985e-05},
    {0.11448871321980414, 0.2119048870388244, 0.11426319305457783, -0.021822737024708799,
     -0.0415077967399776, -0.0071509418838331925, 0.0059140580504170592, 0.0021639136411012697,
     -0.0004333516099163518, -0.00029367746733722713, 1.1535308984768946e-05, 2.4758941012293623e-05},
    {0.37756233506507403, 0.21808286915808384, -0.15846344050821529, -0.10895057581136119,
     0.030015917748356494, 0.02593676442975737, -0.003297963413731838, -0.0039238661577996846,
     0.00021452774175498681, 0.00042401012079782969, -5.6871785827175224e-06, -3.3239772989281143e-05}};

__global__ void __launch_bounds__(kPlanThreads)
k_band_plan(BandReal* __restrict__ dr, BandState* __restrict__ st, const BandReal one,
            bool use_one, int* __restrict__ any_rest) {
  // one grid: its description comes as an argument and is left in dr[0] for
  // the kernels after this one
  if (use_one && threadIdx.x == 0) dr[0] = one;
  band_plan<false>(use_one ? one : dr[blockIdx.x], PointsArgs{}, st + blockIdx.x, any_rest);
}

// ---- work items -------------------------------------------------------------
// Prefix sums of the grids' work items, pre[k][0 .. count] for kernel k (one
// block per kernel; many grids only).
__global__ void __launch_bounds__(kPlanThreads)
k_band_scan(const BandState* __restrict__ st, int count, int64_t* __restrict__ pre) {
  __shared__ int64_t wsum[kPlanThreads / 64];
  const int k = blockIdx.x, tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
  int64_t* out = pre + static_cast<int64_t>(k) * (count + 1);
  int64_t carry = 0;
  for (int base = 0; base < count; base += kPlanThreads) {
    const int64_t v = base + tid < count ? st[base + tid].items[k] : 0;
    int64_t inc = v;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const int64_t y = __shfl_up(inc, o, 64);
      if (lane >= o) inc += y;
    }
    __syncthreads();
    if (lane == 63) wsum[wv] = inc;
    __syncthreads();
    int64_t total = 0;
    for (int w = 0; w < kPlanThreads / 64; ++w) {
      if (w < wv) inc += wsum[w];
      total += wsum[w];
    }
    if (base + tid < count) out[base + tid] = carry + inc - v;
    carry += total;
  }
  if (tid == 0) out[count] = carry;
}

// Work items b, b + nb, .. of kernel k over all grids: f(grid, item in grid).
// pre null: one grid.
template <typename F>
__device__ __forceinline__ void each_item(const BandState* __restrict__ st,
                                          const int64_t* __restrict__ pre, int count, int k, int b,
                                          int nb, F&& f) {
  const int64_t* p = pre ? pre + static_cast<int64_t>(k) * (count + 1) : nullptr;
  const int64_t total = p ? p[count] : st[0].items[k];
  for (int64_t t = b; t < total; t += nb) {
    const int g = p ? find_item(p, count, t) : 0;
    f(g, p ? t - p[g] : t);
  }
}

// ---- weights ---------------------------------------------------------------
// Window weights of the grid's coordinates (block b of nb of a grid); a
// non-finite coordinate gets NaN.
__device__ __forceinline__ void band_weights(const BandReal& R, const BandState& S, int b, int nb) {
  for (int d = 0; d < 3; ++d) {
    if (S.ident[d]) continue;
    const int64_t len = R.len[d];
    for (int64_t i = static_cast<int64_t>(b) * 256 + threadIdx.x; i < len;
         i += static_cast<int64_t>(nb) * 256) {
      const double x = R.ax[d][i];
      int f = 0;
      double r = NAN;
      if (isfinite(x)) {
        const double u = (x - S.lo[d]) / S.h[d];
        f = min(max(static_cast<int>(ceil(u - 0.5 * kBandWidth)), 0), S.n[d] - kBandWidth);
        r = f + (0.5 * kBandWidth - 0.5) - u;
      }
      auto put = [&](int k, double w) {
        if (d == 2) R.wt2[k * len + i] = w;
        else R.wt[d][i * kWeightLd + k] = static_cast<float>(w);
      };
      const double s = r * r;
#pragma unroll
      for (int k = 0; k < kBandWidth / 2; ++k) {
        double e = kTap[k][10], o = kTap[k][11];
#pragma unroll
        for (int j = 4; j >= 0; --j) {
          e = __builtin_fma(e, s, kTap[k][2 * j]);
          o = __builtin_fma(o, s, kTap[k][2 * j + 1]);
        }
        put(k, __builtin_fma(r, o, e));
        put(kBandWidth - 1 - k, __builtin_fma(-r, o, e));
      }
      R.i0[d][i] = f;
    }
  }
}

// ---- node values ------------------------------------------------------------
// F[row][col] = sum_m Im(P(row, m) C(m, col)), row = (i, j) over the nodes of
// the first two axes, P = a e^{2 pi i (kap0 x_i + kap1 y_j + th)}, C = p e^{2
// pi i kap2 z}: a real product over K = 2 modes, (Re P, Im P) against (Im C,
// Re C), as in the factored GEMM (gsc_gemm.h), on v_mfma_f32_32x32x16_f16
// with both operands in two fp16 parts (three products) and the sums in two
// FP32 levels (restarted every 256 modes).  Phases are FP64, reduced exactly,
// then the FP32 sine and cosine instructions: each node carries errors of
// about 1e-7 of a mode, which the interpolation averages over its windows.
// A block of four waves takes TB x TB tiles ((TB / 2)^2 per wave) and one split
// of the modes.  A wave evaluates four modes of each 16-mode chunk (their
// data wave-uniform, in scalar registers) for a row and a column per lane and
// 64; there is no table, since a tile's 2 TB entries per mode cost less than
// reading them would at these sizes.  Bound by that VALU work (TB = 64) or
// about evenly by it and the matrix cores (TB = 128).
constexpr int kNodeLd = 2 * kNodeModes + 8;  // halves per LDS row (80 bytes)
constexpr int kNodeFlush = 16;               // chunks per FP32 accumulation interval

__host__ __device__ __forceinline__ int node_chunks(int n) { return (n + kNodeModes - 1) / kNodeModes; }

__device__ __forceinline__ void split_half(f32x2 v, uint32_t& hi, uint32_t& lo) {
  const half2_t h = __builtin_convertvector(v, half2_t);
  hi = __builtin_bit_cast(uint32_t, h);
  lo = __builtin_bit_cast(uint32_t,
                          __builtin_convertvector(v - __builtin_convertvector(h, f32x2), half2_t));
}

struct NodeSmem {
  _Float16 a[2][128][kNodeLd];
  _Float16 b[2][128][kNodeLd];
};

template <int TB, bool VEC>
__device__ __forceinline__ void node_item(NodeSmem& sm, const BandReal& R, const BandState& S,
                                          int it) {
  constexpr int NB = TB / 64;  // 32 x 32 blocks per wave and side; rows and columns per lane
  const int n1 = S.n[1], n2 = S.n[2];
  const int rows = S.n[0] * n1, cols = n2 * R.ncomp;
  const int ct = (cols + TB - 1) / TB;
  const int chunks = node_chunks(S.n_in);
  const int lane = threadIdx.x & 63, hl = lane >> 5, lr = lane & 31;
  const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wr = TB / 2 * (wv >> 1), wc = TB / 2 * (wv & 1);
  const int ae = S.amp_exp;  // (as a factor it may not be finite)
  const auto bm = const_ptr(R.bm);
  auto node = [&](int d, int i) { return S.ident[d] ? R.ax[d][i] : S.lo[d] + i * S.h[d]; };
  const int sp = it % S.splits, tile = it / S.splits;
  const int r0 = tile / ct * TB, c0 = tile % ct * TB;
  const int q0 = static_cast<int>(static_cast<int64_t>(chunks) * sp / S.splits);
  const int q1 = static_cast<int>(static_cast<int64_t>(chunks) * (sp + 1) / S.splits);
  // this lane's rows and columns (clamped: those past the end are not stored)
  double x[NB], y[NB], z[NB];
  int comp[NB];
#pragma unroll
  for (int u = 0; u < NB; ++u) {
    const int row = min(r0 + lane + 64 * u, rows - 1), col = min(c0 + lane + 64 * u, cols - 1);
    const int ri = row / n1, cc = col / n2;
    x[u] = node(0, ri);
    y[u] = R.dim == 3 ? node(1, row - ri * n1) : 0.0;
    z[u] = node(2, col - cc * n2);
    comp[u] = cc;
  }
  // the wave's four modes of a chunk, read (scalar loads) a chunk ahead
  struct Quad {
    double k0[4], k1[4], k2[4], th[4];
    float am[4], pr[VEC ? 4 : 1][3];
  } md;
  auto load = [&](int q) {
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const auto p = bm + q * kNodeModes + 4 * wv + e;
      md.k0[e] = p->kap[0];
      md.k1[e] = p->kap[1];
      md.k2[e] = p->kap[2];
      md.th[e] = p->th;
      md.am[e] = p->amp;
      if constexpr (VEC)
#pragma unroll
        for (int c = 0; c < 3; ++c) md.pr[e][c] = p->proj[c];
    }
  };
  f32x16 acc[NB][NB], tot[NB][NB];
#pragma unroll
  for (int i = 0; i < NB; ++i)
#pragma unroll
    for (int j = 0; j < NB; ++j)
#pragma unroll
      for (int v = 0; v < 16; ++v) tot[i][j][v] = 0.0f;
  load(q0);
  for (int qb = q0; qb < q1; qb += kNodeFlush) {
#pragma unroll
    for (int i = 0; i < NB; ++i)
#pragma unroll
      for (int j = 0; j < NB; ++j)
#pragma unroll
        for (int v = 0; v < 16; ++v) acc[i][j][v] = 0.0f;
    const int qe = min(qb + kNodeFlush, q1);
    for (int q = qb; q < qe; ++q) {
      uint32_t ph[NB][4], pl[NB][4], ch[NB][4], cl[NB][4];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const float a = __builtin_ldexpf(md.am[e], ae);
#pragma unroll
        for (int u = 0; u < NB; ++u) {
          const double t = __builtin_fma(md.k1[e], y[u], __builtin_fma(md.k0[e], x[u], md.th[e]));
          const float r = static_cast<float>(t - rint(t));
          split_half(f32x2{a * __builtin_amdgcn_cosf(r), a * __builtin_amdgcn_sinf(r)}, ph[u][e],
                     pl[u][e]);
          const double tz = md.k2[e] * z[u];
          const float rz = static_cast<float>(tz - rint(tz));
          f32x2 c{__builtin_amdgcn_sinf(rz), __builtin_amdgcn_cosf(rz)};
          if constexpr (VEC)
            c = c * (comp[u] == 0 ? md.pr[e][0] : (comp[u] == 1 ? md.pr[e][1] : md.pr[e][2]));
          split_half(c, ch[u][e], cl[u][e]);
        }
      }
      __syncthreads();  // the previous chunk is read
#pragma unroll
      for (int u = 0; u < NB; ++u) {
        const int l = lane + 64 * u;
        *reinterpret_cast<u32x4*>(&sm.a[0][l][8 * wv]) = u32x4{ph[u][0], ph[u][1], ph[u][2], ph[u][3]};
        *reinterpret_cast<u32x4*>(&sm.a[1][l][8 * wv]) = u32x4{pl[u][0], pl[u][1], pl[u][2], pl[u][3]};
        *reinterpret_cast<u32x4*>(&sm.b[0][l][8 * wv]) = u32x4{ch[u][0], ch[u][1], ch[u][2], ch[u][3]};
        *reinterpret_cast<u32x4*>(&sm.b[1][l][8 * wv]) = u32x4{cl[u][0], cl[u][1], cl[u][2], cl[u][3]};
      }
      __syncthreads();
      load(min(q + 1, q1 - 1));
#pragma unroll
      for (int ks = 0; ks < 2; ++ks) {
        half8 fa[2][NB], fb[2][NB];
#pragma unroll
        for (int p = 0; p < 2; ++p)
#pragma unroll
          for (int i = 0; i < NB; ++i) {
            fa[p][i] = *reinterpret_cast<const half8*>(&sm.a[p][wr + 32 * i + lr][16 * ks + 8 * hl]);
            fb[p][i] = *reinterpret_cast<const half8*>(&sm.b[p][wc + 32 * i + lr][16 * ks + 8 * hl]);
          }
#pragma unroll
        for (int s = 0; s < 3; ++s)  // hi hi, hi lo, lo hi
#pragma unroll
          for (int i = 0; i < NB; ++i)
#pragma unroll
            for (int j = 0; j < NB; ++j)
              acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(fa[s == 2][i], fb[s == 1][j],
                                                                 acc[i][j], 0, 0, 0);
      }
    }
#pragma unroll
    for (int i = 0; i < NB; ++i)
#pragma unroll
      for (int j = 0; j < NB; ++j)
#pragma unroll
        for (int v = 0; v < 16; ++v) tot[i][j][v] += acc[i][j][v];
  }
  float* F = R.F + static_cast<int64_t>(sp) * rows * cols;
#pragma unroll
  for (int i = 0; i < NB; ++i)
#pragma unroll
    for (int j = 0; j < NB; ++j)
#pragma unroll
      for (int v = 0; v < 16; ++v) {
        const int r = r0 + wr + 32 * i + 8 * (v >> 2) + 4 * hl + (v & 3);
        const int c = c0 + wc + 32 * j + lr;
        if (r < rows && c < cols) F[static_cast<int64_t>(r) * cols + c] = tot[i][j][v];
      }
}

__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2, 2)))
k_band_nodes(const BandReal* __restrict__ dr, const BandState* __restrict__ st,
             const int64_t* __restrict__ pre, int count, int wblocks, int nblocks, int rblocks,
             const TableArgs ta) {
  __shared__ __attribute__((aligned(16))) NodeSmem sm;
  const int b = blockIdx.x;  // every branch on it is uniform over the block
  if (b >= wblocks + nblocks) {
    // tables of the rest modes (one grid): 64 rows of one chunk and role
    const int e = b - wblocks - nblocks, rc = e / rblocks, m = st[0].n_rest;
    if (rc / 3 < mode_chunks(m))
      gemm::table_quad<_Float16, 2>(ta.modes, m, ta.dim, ta.nch, ta.xs, ta.xa, ta.xc, ta.na,
                                    ta.nrow, ta.arows, ta.ncols, ta.ncp, ta.S, ta.A, ta.C, rc % 3,
                                    static_cast<int64_t>(e % rblocks) * 64 + (threadIdx.x & 63),
                                    rc / 3, threadIdx.x >> 6, ta.trans, ta.ncomp, ta.pg);
    return;
  }
  if (b < wblocks) {  // shared evenly by the grids
    const int per = wblocks / count, g = b / per;
    const BandState S = st[g];
    if (S.n_in > 0) band_weights(dr[g], S, b - g * per, per);
    return;
  }
  each_item(st, pre, count, 0, b - wblocks, nblocks, [&](int g, int64_t it) {
    const BandState S = st[g];
    const int i = static_cast<int>(it);
    if (dr[g].ncomp > 1) {
      if (S.big) node_item<128, true>(sm, dr[g], S, i);
      else node_item<64, true>(sm, dr[g], S, i);
    } else {
      if (S.big) node_item<128, false>(sm, dr[g], S, i);
      else node_item<64, false>(sm, dr[g], S, i);
    }
  });
}

// ---- interpolation ------------------------------------------------------------
// Last axis: t1[comp][row][c] from the nodes of row (FP64 sums, splits added
// in order).  An item is up to last_rows (row, comp) lines, which share a
// column's weights; the lines' nodes pass through LDS, as many lines at a
// time as fit.
constexpr int kLineMax = 2048;  // nodes held in LDS (one line at least)
__global__ void __launch_bounds__(256)
k_band_last(const BandReal* __restrict__ dr, const BandState* __restrict__ st,
            const int64_t* __restrict__ pre, int count) {
  __shared__ double line[kLineMax];
  const int tid = threadIdx.x;
  each_item(st, pre, count, 1, blockIdx.x, gridDim.x, [&](int gi, int64_t it) {
    const BandReal& R = dr[gi];
    const BandState S = st[gi];
    const int rows = S.n[0] * S.n[1], n2 = S.n[2], cols = n2 * R.ncomp;
    const int len = static_cast<int>(R.len[2]);
    const int64_t fs = static_cast<int64_t>(rows) * cols;
    const auto wt = global_ptr(R.wt2);
    const auto i0 = global_ptr(R.i0[2]);
    const auto F = global_ptr(R.F);
    const auto t1 = global_ptr(R.t1);
    const int l1 = min((static_cast<int>(it) + 1) * S.last_rows, rows * R.ncomp);
    const int fit = min(kLineMax / n2, S.last_rows);
    for (int l = static_cast<int>(it) * S.last_rows; l < l1; l += fit) {
      const int nl = min(fit, l1 - l);
      __syncthreads();  // the previous lines are read
      for (int e = tid; e < nl * n2; e += 256) {
        const int li = l + e / n2, comp = li / rows;
        const int64_t f0 =
            static_cast<int64_t>(li - comp * rows) * cols + comp * n2 + (e - e / n2 * n2);
        double v = 0.0;
#pragma unroll 4
        for (int s = 0; s < S.splits; ++s) v += static_cast<double>(F[s * fs + f0]);
        line[e] = v * S.out_scale;
      }
      __syncthreads();
      for (int c = tid; c < len; c += 256) {
        double w[kBandWidth];
        int f = c;
        if (!S.ident[2]) {  // uniform
          f = i0[c];
#pragma unroll
          for (int k = 0; k < kBandWidth; ++k) w[k] = wt[static_cast<int64_t>(k) * len + c];
        }
        for (int j = 0; j < nl; ++j) {
          const double* p = line + j * n2 + f;
          double v = 0.0;
          if (S.ident[2]) {
            v = p[0];
          } else {
#pragma unroll
            for (int k = 0; k < kBandWidth; ++k) v = __builtin_fma(w[k], p[k], v);
          }
          t1[static_cast<int64_t>(l + j) * len + c] = static_cast<float>(v);
        }
      }
    }
  });
}

// One axis in FP32: out[p][q] (p over the axis' coordinates) from in[node][q].
// An item is a run of coordinates by a block's columns; a lane takes C of
// them: q .. q + 3 in one 16-byte access (C = 4; VEC 1: aligned, 2: at any
// word), or q + 256 c (VEC 0).  It keeps
// the window of nodes in registers while p walks over the run, reading one
// node ahead; the run's weights and window places pass through LDS.  ADD:
// out += (the factored GEMM's part is there).  Bound by the output's bytes on
// fine meshes.
constexpr int kMaxRun = kFirstRunShared;
static_assert(kMidRun <= kMaxRun && kFirstRun <= kMaxRun, "runs");
struct RunSmem {
  f32x4 w[kMaxRun][kBandWidth / 4];
  int f[kMaxRun];
};
static_assert(kWeightLd == kBandWidth && kBandWidth % 4 == 0, "weights in whole vectors");

// (barriers: the whole block)
__device__ __forceinline__ void run_weights(RunSmem& sm, const float* weights, const int* first,
                                            int64_t p0, int64_t p1) {
  __syncthreads();  // the previous run is read
  const int n = static_cast<int>(p1 - p0);
  const auto w = global_ptr(reinterpret_cast<const f32x4*>(weights + p0 * kWeightLd));
  for (int e = threadIdx.x; e < n * (kBandWidth / 4); e += 256) (&sm.w[0][0])[e] = w[e];
  for (int e = threadIdx.x; e < n; e += 256) sm.f[e] = global_ptr(first)[p0 + e];
  __syncthreads();
}

template <int C, int VEC, bool ADD, typename InP, typename OutP>
__device__ __forceinline__ void band_run(const RunSmem& sm, InP in, OutP out, int64_t width,
                                         int nodes, int ident, unsigned q, int64_t p0, int n) {
  static_assert(VEC == 0 || C == 4, "one 16-byte access");
  static_assert(VEC != 2 || !ADD, "overlapping lanes do not add");
  typedef float T __attribute__((ext_vector_type(C)));
  typedef float TM __attribute__((ext_vector_type(C), aligned(VEC == 2 ? 4 : sizeof(T))));
  using GT = __attribute__((address_space(1))) TM;
  // rows are uniform pointers, the lane's columns 32-bit offsets
  auto get = [&](int row) {
    const auto p = in + row * width;
    T v;
    if constexpr (VEC != 0) {
      v = *reinterpret_cast<const GT*>(p + q);
    } else {
#pragma unroll
      for (int c = 0; c < C; ++c) v[c] = p[q + 256u * c];
    }
    return v;
  };
  OutP row = out + p0 * width;
  auto put = [&](T v) {
    if constexpr (VEC != 0) {
      auto* o = reinterpret_cast<GT*>(row + q);
      if constexpr (VEC == 1 && !ADD) __builtin_nontemporal_store(v, o);
      else *o = v;  // (rows start anywhere: L2 joins their ends)
    } else {
#pragma unroll
      for (int c = 0; c < C; ++c) row[q + 256u * c] = v[c];
    }
    row += width;
  };
  // the window, and the node after it, read ahead of the move that needs it
  T win[kBandWidth], nxt;
  int cur = -(1 << 30);
  auto value = [&](int i) {
    if (ident) return get(static_cast<int>(p0) + i);
    const int fn = __builtin_amdgcn_readfirstlane(sm.f[i]);
    if (fn != cur) {  // uniform
      if (fn == cur + 1) {
#pragma unroll
        for (int k = 0; k + 1 < kBandWidth; ++k) win[k] = win[k + 1];
        win[kBandWidth - 1] = nxt;
      } else {
#pragma unroll
        for (int k = 0; k < kBandWidth; ++k) win[k] = get(fn + k);
      }
      nxt = get(min(fn + kBandWidth, nodes - 1));
      cur = fn;
    }
    T v = win[0] * sm.w[i][0][0];
#pragma unroll
    for (int k = 1; k < kBandWidth; ++k)
#pragma unroll
      for (int c = 0; c < C; ++c) v[c] = __builtin_fmaf(win[k][c], sm.w[i][k / 4][k % 4], v[c]);
    return v;
  };
  if constexpr (!ADD) {
    for (int i = 0; i < n; ++i) put(value(i));
  } else {
    // what the GEMM left is read kAhead rows at a time: read row by row it
    // would wait for the stores before
    constexpr int kAhead = 4;
    for (int i0 = 0; i0 < n; i0 += kAhead) {
      T old[kAhead];
#pragma unroll
      for (int u = 0; u < kAhead; ++u) {
        const auto o = row + min(u, n - 1 - i0) * width;
        if constexpr (VEC != 0) {
          old[u] = *reinterpret_cast<const GT*>(o + q);
        } else {
#pragma unroll
          for (int c = 0; c < C; ++c) old[u][c] = o[q + 256u * c];
        }
      }
#pragma unroll
      for (int u = 0; u < kAhead; ++u)
        if (i0 + u < n) put(old[u] + value(i0 + u));
    }
  }
}

// Middle axis of a 3-D grid: t2[comp][i][b][c] from t1[comp][i][j][c].
__global__ void __launch_bounds__(256)
k_band_mid(const BandReal* __restrict__ dr, const BandState* __restrict__ st,
           const int64_t* __restrict__ pre, int count) {
  __shared__ RunSmem sm;
  each_item(st, pre, count, 2, blockIdx.x, gridDim.x, [&](int gi, int64_t it) {
    const BandReal& R = dr[gi];
    const BandState S = st[gi];
    const int64_t len = R.len[1], width = R.len[2];
    const int64_t qb = (width + 255) / 256, pb = (len + kMidRun - 1) / kMidRun;
    const int64_t plane = it / (qb * pb), r = it - plane * (qb * pb);
    const unsigned q = static_cast<unsigned>(r % qb) * 256 + threadIdx.x;
    const int64_t p0 = r / qb * kMidRun, p1 = min(p0 + kMidRun, len);
    if (!S.ident[1]) run_weights(sm, R.wt[1], R.i0[1], p0, p1);
    if (q < width)
      band_run<1, 0, false>(sm, global_ptr(R.t1) + plane * S.n[1] * width,
                                global_ptr(R.t2) + plane * len * width, width, S.n[1], S.ident[1],
                                q, p0, static_cast<int>(p1 - p0));
  });
}

// First axis, into the output.
template <int C, int VEC>
__device__ __forceinline__ void first_run(const RunSmem& sm, const BandReal& R, const BandState& S,
                                          int64_t comp, unsigned q, int64_t p0, int n) {
  const int64_t width = R.len[1] * R.len[2];
  const auto in = global_ptr(R.dim == 3 ? R.t2 : R.t1) + comp * S.n[0] * width;
  const auto out = global_ptr(R.out) + comp * R.len[0] * width;
  if constexpr (VEC != 2) {
    if (S.n_rest > 0) {  // uniform
      band_run<C, VEC, true>(sm, in, out, width, S.n[0], S.ident[0], q, p0, n);
      return;
    }
  }
  band_run<C, VEC, false>(sm, in, out, width, S.n[0], S.ident[0], q, p0, n);
}
__global__ void __launch_bounds__(256)
k_band_first(const BandReal* __restrict__ dr, const BandState* __restrict__ st,
             const int64_t* __restrict__ pre, int count) {
  __shared__ RunSmem sm;
  each_item(st, pre, count, 3, blockIdx.x, gridDim.x, [&](int gi, int64_t it) {
    const BandReal& R = dr[gi];
    const BandState S = st[gi];
    const int64_t len = R.len[0], width = R.len[1] * R.len[2];
    const int64_t qc = 256 * S.first_cols, qb = (width + qc - 1) / qc;
    const int64_t pb = (len + S.first_run - 1) / S.first_run;
    const int64_t comp = it / (qb * pb), r = it - comp * (qb * pb);
    const int64_t p0 = r / qb * S.first_run, p1 = min(p0 + S.first_run, len);
    if (!S.ident[0]) run_weights(sm, R.wt[0], R.i0[0], p0, p1);
    const int n = static_cast<int>(p1 - p0);
    const int64_t q = (r % qb) * qc + (S.vec ? 4 * threadIdx.x : threadIdx.x);
    if (q >= width) return;
    const unsigned qu = static_cast<unsigned>(q);
    if (S.vec == 1) {
      first_run<4, 1>(sm, R, S, comp, qu, p0, n);
      return;
    }
    if (S.vec == 2) {
      first_run<4, 2>(sm, R, S, comp, min(qu, static_cast<unsigned>(width) - 4u), p0, n);
      return;
    }
    // the lane's columns that exist (first_cols or one less)
    const int64_t nc = min((width - q + 255) / 256, static_cast<int64_t>(S.first_cols));
    if (nc == 4) first_run<4, 0>(sm, R, S, comp, qu, p0, n);
    else if (nc == 3) first_run<3, 0>(sm, R, S, comp, qu, p0, n);
    else if (nc == 2) first_run<2, 0>(sm, R, S, comp, qu, p0, n);
    else first_run<1, 0>(sm, R, S, comp, qu, p0, n);
  });
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
    // at most three fifths as many nodes as coordinates, or all of a short axis
    const int64_t c = std::min<int64_t>(p.len[d], p.len[d] * 3 / 5 + kBandWidth + 2);
    p.cap[d] = static_cast<int>(std::min<int64_t>(c, d == 2 ? kLineMax : 1 << 20));
  }
  if (dim == 3) {
    const int64_t plane = p.len[1] * p.len[2] * ncomp;
    p.cap[0] = static_cast<int>(std::min<int64_t>(p.cap[0], kT2Max / plane));
  }
  // (more nodes than a third of the grid's points never pay)
  p.fcap = std::max<int64_t>(N * ncomp / 3, 1 << 16);
  const int64_t rows = static_cast<int64_t>(p.cap[0]) * p.cap[1];
  const int64_t t1max = std::min<int64_t>(rows, p.fcap) * p.len[2] * ncomp;
  p.on = p.len[1] * p.len[2] < (int64_t(1) << 30) && p.cap[0] > 0 && p.fcap < (int64_t(1) << 31) && t1max < (int64_t(1) << 29);
  if (!p.on) return p;
  size_t off = 0;
  auto take = [&off](size_t b) {
    const size_t o = off;
    off += (b + 255) & ~static_cast<size_t>(255);
    return o;
  };
  p.rest = take(sizeof(ModeRec) * static_cast<size_t>(M));
  p.bm = take(sizeof(BandMode) * static_cast<size_t>(M + kNodeModes));
  for (int d = 0; d < 3; ++d) {
    if (dim == 2 && d == 1) continue;
    p.i0[d] = take(sizeof(int) * static_cast<size_t>(p.len[d]));
    p.wt[d] = take((d == 2 ? sizeof(double) * kBandWidth : sizeof(float) * kWeightLd) *
                   static_cast<size_t>(p.len[d]));
  }
  p.F = take(sizeof(float) * static_cast<size_t>(p.fcap));
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
  r->bm = reinterpret_cast<BandMode*>(b + p.bm);
  for (int d = 0; d < 3; ++d) {
    r->len[d] = p.len[d];
    r->cap[d] = p.cap[d];
    r->i0[d] = reinterpret_cast<int*>(b + p.i0[d]);
    r->wt[d] = reinterpret_cast<float*>(b + p.wt[d]);
  }
  r->wt2 = reinterpret_cast<double*>(b + p.wt[2]);
  r->F = reinterpret_cast<float*>(b + p.F);
  r->t1 = reinterpret_cast<float*>(b + p.t1);
  r->t2 = reinterpret_cast<float*>(b + p.t2);
}

hipError_t launch_band_plan(const BandLaunch& L, const BandReal* one, const TableArgs* rest,
                            hipStream_t s) {
  const int count = L.count;
  k_band_plan<<<count, kPlanThreads, 0, s>>>(L.d, L.st, one ? *one : BandReal{}, one != nullptr,
                                             L.any_rest);
  if (L.pre) k_band_scan<<<kBandLists, kPlanThreads, 0, s>>>(L.st, count, L.pre);
  // blocks for the weights, the node tiles and the rest modes' tables
  const int wb = L.pre ? count * std::min(std::max(256 / count, 1), 4) : 16, nb = 1024;
  const int64_t rb = rest ? table_row_blocks(*rest, true) : 1;
  const int64_t tb = rest ? rb * 3 * rest->nch : 0;
  k_band_nodes<<<static_cast<unsigned>(wb + nb + tb), 256, 0, s>>>(
      L.d, L.st, L.pre, count, wb, nb, static_cast<int>(rb), rest ? *rest : TableArgs{});
  return hipGetLastError();
}

hipError_t launch_band_plans(const BandLaunch& L, hipStream_t s) {
  k_band_plan<<<L.count, kPlanThreads, 0, s>>>(L.d, L.st, BandReal{}, false, L.any_rest);
  return hipGetLastError();
}

// Seconds in a replayed graph, measured on one MI355X over plans of 32 to 1024 modes:
// a chunk of 16 modes of a 256 x 128 tile in a full round of tiles and of a
// realisation's tables; of the longest tables and tiles where there are few; the
// kernels' own time; and the band's launches (plan 12 to 16, scan 5, nodes 6, last and
// first axis 5 each).  Without and with the band: 3 realisations of 206 exponential
// modes 52 and 84 us, 181 of 255 271 and 352, 444 of 355 408 and 310, 10 of 203
// Gaussian modes 82 and 48.
constexpr double kEnsChunk = 1.45e-6, kEnsTableChunk = 17e-9;
constexpr double kEnsTableAlone = 0.5e-6, kEnsChunkAlone = 1.1e-6;
constexpr double kEnsTables = 10e-6, kEnsGemm = 12e-6, kEnsBand = 33e-6;
bool band_ensemble_pays(const BandReal* r, const BandState* st, int count, int gemms,
                        const EnsChunks& other) {
  EnsChunks off = other, on = other;
  double band = 0.0, node = 0.0, node_chain = 0.0;
  for (int i = 0; i < count; ++i) {
    const BandState& s = st[i];
    const int all = mode_chunks(r[i].M);
    off.add(r[i].gemm_tiles, all);
    on.add(r[i].gemm_tiles, s.n_in > 0 ? mode_chunks(s.n_rest) : all);
    if (s.n_in <= 0) continue;
    const float rows = static_cast<float>(s.n[0]) * s.n[1];
    bool big;
    const int chunks = node_chunks(s.n_in);
    node += node_tiles(rows, static_cast<float>(s.n[2]) * r[i].ncomp, true, big) * chunks / kCus;
    node_chain = std::max(node_chain, static_cast<double>(kNodeChunkAlone) * chunks / s.splits);
    const double n1 = static_cast<double>(r[i].len[1]), n2 = static_cast<double>(r[i].len[2]);
    const double stream = 2.0 * rows * n2 + (r[i].dim == 3 ? 2.0 * s.n[0] * n1 * n2 : 0.0);
    const double out = static_cast<double>(r[i].len[0]) * n1 * n2 * (s.n_rest > 0 ? 3.0 : 1.0);
    band += (stream + out) * r[i].ncomp * (4.0 * kStreamByte);
  }
  auto gemm = [gemms](const EnsChunks& c) {
    if (c.longest == 0) return 0.0;
    return std::max(c.tiles * kEnsChunk / kCus + c.tables * kEnsTableChunk,
                    c.longest * (kEnsTableAlone + gemms * kEnsChunkAlone)) +
           kEnsTables + gemms * kEnsGemm;
  };
  return kEnsBand + band + std::max(node, node_chain) + gemm(on) < gemm(off);
}

hipError_t launch_band_nodes(const BandLaunch& L, hipStream_t s) {
  k_band_nodes<<<1024, 256, 0, s>>>(L.d, L.st, nullptr, 1, 0, 1024, 1, TableArgs{});
  return hipGetLastError();
}

hipError_t launch_band_finish(const BandLaunch& L, hipStream_t s) {
  k_band_last<<<2048, 256, 0, s>>>(L.d, L.st, L.pre, L.count);
  if (L.dim == 3) k_band_mid<<<4096, 256, 0, s>>>(L.d, L.st, L.pre, L.count);
  k_band_first<<<4096, 256, 0, s>>>(L.d, L.st, L.pre, L.count);
  return hipGetLastError();
}

}  // namespace gsc
