// Band-limited evaluation of fields at point lists (3-D, float32 results).
//
// As band.hip for grids: the modes with |kap_d| <= K_d are summed on a coarse
// uniform grid of nodes and interpolated with the same window, here point by
// point over 8 x 8 x 8 nodes.  The points are cell-sorted as for the local
// kernel (direct_local.hip), in cells so small that a cell's points share one
// window of 10, 12 or 16 x 16 x 16 nodes (cells at most 1.9, 3.9 or 7.9 x 7.9 x 6.9
// nodes wide), and the interpolation along the last axis is a matrix product: rows
// the window's (i, j) lines, K its 16 nodes along the line, columns 32 points'
// weights.  The other two axes are multiply-adds on the products, 18 per lane and
// tile of 32 x 32.  Modes outside the band are summed per point with FP64 phases by
// the launch that would have run the local kernel (band_rest).
#include "gsc_band.h"
#include "gsc_band_plan.h"
#include "gsc_device.h"
#include "gsc_local.h"

#include <hip/hip_runtime.h>

#include <algorithm>

namespace gsc {
namespace {

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef u32x4 u32x4u __attribute__((aligned(4)));

__device__ __forceinline__ void half_parts(float v, _Float16& h, _Float16& l) {
  h = static_cast<_Float16>(v);
  l = static_cast<_Float16>(v - static_cast<float>(h));
}

// Node values: the splits added in order (FP64), scaled, in two fp16 parts.  (By
// the node kernel's last block of a tile instead, 110 us more: the fences that
// needs write each die's L2 back.)
__global__ void __launch_bounds__(256)
k_band_sum(const BandReal* __restrict__ dr, const BandState* __restrict__ st,
           _Float16* __restrict__ G, int64_t gl) {
  const BandState S = *st;
  if (S.n_in == 0) return;
  const int64_t n = static_cast<int64_t>(S.n[0]) * S.n[1] * S.n[2] * dr->ncomp;
  const auto F = global_ptr(dr->F);
  for (int64_t e = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x; e < n;
       e += static_cast<int64_t>(gridDim.x) * 256) {
    double v = 0.0;
#pragma unroll 4
    for (int s = 0; s < S.splits; ++s) v += static_cast<double>(F[s * n + e]);
    float f = static_cast<float>(v * S.g_scale);
    __asm__ volatile("" : "+v"(f));  // FP32 rounding step kept
    half_parts(f, G[e], G[gl + e]);
  }
}

// The window's taps at distances 3.5 - k - r (k < 4) as polynomials in r over
// |r| <= 1/2, and at k - 3.5 - r with -r: Chebyshev fits of
// I0(beta sqrt(1 - (2 u / 8)^2)) / c0 to 3e-9 (5e-8 with the roundings).
constexpr int kTapCoef = 9;
constexpr float kTap[4][kTapCoef] = {
    {3.777812753e-05f, 3.035890170e-04f, 1.043527902e-03f, 2.006990965e-03f, 2.354347876e-03f,
     1.686687085e-03f, 6.311407620e-04f, -2.300197108e-05f, -1.127378819e-04f},
    {7.911188892e-03f, 2.881554561e-02f, 4.315619654e-02f, 3.207364048e-02f, 9.141288423e-03f,
     -3.256056079e-03f, -3.251838055e-03f, -4.709302619e-04f, 3.109832679e-04f},
    {1.144887132e-01f, 2.119049253e-01f, 1.142631887e-01f, -2.182478409e-02f, -4.150765593e-02f,
     -7.121297914e-03f, 5.912480957e-03f, 2.004039369e-03f, -4.261420410e-04f},
    {3.775623351e-01f, 2.180828137e-01f, -1.584634383e-01f, -1.089476097e-01f, 3.001584832e-02f,
     2.589382995e-02f, -3.297185870e-03f, -3.692501822e-03f, 2.109732558e-04f}};

static_assert(kWinCols == 16, "a tile is two planes of 16 lines");
constexpr float kTapScale = 256.0f;  // of the fp16 weights (parts clear of subnormals)
// LDS row of a point's dense weights: fp16 parts of the last axis', the middle
// and the first axis' (bytes)
constexpr int kRowY = 64, kRowX = 128;
constexpr int row_bytes(int tiles) { return kRowX + (2 * tiles + 3) / 4 * 16; }
constexpr int kRowMax = row_bytes(8);

// A wave takes record groups (64 points, one cell) from a contiguous share; a
// component's window is in registers as fp16 fragments.  Fragment of
// tile t: row r = lane % 32 is line i = 2 t + r / 16, j = r % 16 of the window, K
// slots its nodes 8 hl .. 8 hl + 7 (hl = lane / 32).  A half group's 32 points
// are the columns; the points' dense weights (8 taps among 16 slots, zero
// elsewhere), one point per lane, pass through LDS rows.  Product element v of a lane is line (i, j) = (2 t + v / 8, 8 ((v / 4) %
// 2) + 4 hl + v % 4) at point lane % 32.
// Bound by its instructions, which matrix ones hardly overlap: of 49 us for 2e6
// points (five tiles), 15 are 30 matrix instructions of 32 cycles per group, 33
// the vector ones (18 per tile and half group, the taps, their split).  Tried:
// a wave per block, 8192 or 16384 of them: 62 and 64 us; five tiles at two waves
// per SIMD, 64 us; taps per half group by both lanes of a point, 65 us; the
// three components' windows read again per group, 505 us for 4e6 points, 268 us
// in registers (202 us with the places in fixed point and shorter tap
// polynomials; more than five tiles leave no room for them).
// RELOAD: the windows of a vector field's components do not fit in registers
// together and are read again for every group.
template <int NC, int TILES, bool RELOAD>
__device__ __forceinline__ void points_run(char* rows, const BinParams* __restrict__ prm,
                                           const BandState* __restrict__ st,
                                           const _Float16* __restrict__ G, int64_t gl,
                                           const double* __restrict__ centre,
                                           const int* __restrict__ wave_cell, float4* recs,
                                           bool in_place, float* __restrict__ out,
                                           int64_t out_ld) {
  constexpr int kRowLd = row_bytes(TILES);
  constexpr int kRows = 2 * TILES;
  const int lane = threadIdx.x & 63, hl = lane >> 5, lr = lane & 31;
  const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int64_t nw = prm->nwaves, nwv = static_cast<int64_t>(gridDim.x) * 4;
  const int64_t w = static_cast<int64_t>(blockIdx.x) * 4 + wv;
  const int g0 = static_cast<int>(nw * w / nwv), g1 = static_cast<int>(nw * (w + 1) / nwv);
  const int n1 = st->n[1], n2 = st->n[2];
  const int cols = n2 * NC;
  const double oscale = st->out_scale / kTapScale;
  rows += wv * (kWavePts * kRowLd);
  char* row = rows + lane * kRowLd;
  constexpr int NW = RELOAD ? 1 : NC;
  half8 ah[NW][TILES], al[NW][TILES];
  int base[3] = {0, 0, 0};
  // component c's window (the last axis' place is even: whole words)
  auto window = [&](int c) {
    const int w = RELOAD ? 0 : c;
#pragma unroll
    for (int t = 0; t < TILES; ++t) {
      const int64_t line =
          static_cast<int64_t>(base[0] + 2 * t + (lr >> 4)) * n1 + base[1] + (lr & 15);
      const auto p = global_ptr(G + line * cols + c * n2 + base[2] + 8 * hl);
      using GV = const __attribute__((address_space(1))) u32x4u;
      ah[w][t] = __builtin_bit_cast(half8, static_cast<u32x4>(*(GV*)(p)));
      al[w][t] = __builtin_bit_cast(half8, static_cast<u32x4>(*(GV*)(p + gl)));
    }
  };
  int cur = -1;
  if (g0 >= g1) return;
  // the next group's record and cell are read ahead
  float4 rec_next = recs[static_cast<int64_t>(g0) * kWavePts + lane];
  int cell_next = wave_cell[g0];
  for (int g = g0; g < g1; ++g) {
    const float4 rec = rec_next;
    const int cell = __builtin_amdgcn_readfirstlane(cell_next);
    {
      const int gn = min(g + 1, g1 - 1);
      rec_next = recs[static_cast<int64_t>(gn) * kWavePts + lane];
      cell_next = wave_cell[gn];
    }
    if (cell != cur) {  // uniform
      cur = cell;
#pragma unroll
      for (int d = 0; d < 3; ++d)
        base[d] = window_base(*prm, d, centre[4 * static_cast<int64_t>(cell) + d]);
      if constexpr (!RELOAD)
#pragma unroll
        for (int c = 0; c < NC; ++c) window(c);
    }
    // dense weights of the lane's point
    const int idx = __builtin_bit_cast(int, rec.w);
    const float place[3] = {rec.x, rec.y, rec.z};
    __asm__ volatile("" ::: "memory");
#pragma unroll
    for (int i = 0; i < kRowLd; i += 16) *reinterpret_cast<f32x4*>(row + i) = f32x4{};
    __asm__ volatile("" ::: "memory");
#pragma unroll
    for (int d = 0; d < 3; ++d) {
      // (padding: anything in range)
      const uint32_t q = __builtin_bit_cast(uint32_t, place[d]);
      const float r = __builtin_fmaf(static_cast<float>(q & kPlaceMask),
                                     static_cast<float>(1.0 / kPlaceUnit), -0.5f);
      char* rd = row + (d == 0 ? kRowX : (d == 1 ? kRowY : 0)) + (q >> 28) * (d == 2 ? 2u : 4u);
      auto put = [&](int k, float w) {
        if (d == 2) {
          _Float16 h, l;
          half_parts(w * kTapScale, h, l);
          *reinterpret_cast<_Float16*>(rd + 2 * k) = h;
          *reinterpret_cast<_Float16*>(rd + 32 + 2 * k) = l;
        } else {
          *reinterpret_cast<float*>(rd + 4 * k) = w;
        }
      };
      const float s = r * r;
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        float e = kTap[k][8], o = kTap[k][7];
#pragma unroll
        for (int i = 3; i >= 0; --i) e = __builtin_fmaf(e, s, kTap[k][2 * i]);
#pragma unroll
        for (int i = 2; i >= 0; --i) o = __builtin_fmaf(o, s, kTap[k][2 * i + 1]);
        put(k, __builtin_fmaf(r, o, e));
        put(7 - k, __builtin_fmaf(-r, o, e));
      }
    }
    __asm__ volatile("" ::: "memory");
    float res[NC];
#pragma unroll
    for (int c = 0; c < NC; ++c) {
      if constexpr (RELOAD) window(c);
      const int w = RELOAD ? 0 : c;
#pragma unroll
      for (int half = 0; half < 2; ++half) {
        const char* rp = rows + (32 * half + lr) * kRowLd;
        const half8 bh = *reinterpret_cast<const half8*>(rp + 16 * hl);
        const half8 bl = *reinterpret_cast<const half8*>(rp + 32 + 16 * hl);
        float wy[8], wx[(kRows + 3) / 4 * 4];
#pragma unroll
        for (int q = 0; q < 2; ++q) {
          const f32x4 y = *reinterpret_cast<const f32x4*>(rp + kRowY + 32 * q + 16 * hl);
#pragma unroll
          for (int i = 0; i < 4; ++i) wy[4 * q + i] = y[i];
        }
#pragma unroll
        for (int q = 0; q < (kRows + 3) / 4; ++q) {
          const f32x4 x = *reinterpret_cast<const f32x4*>(rp + kRowX + 16 * q);
#pragma unroll
          for (int i = 0; i < 4; ++i) wx[4 * q + i] = x[i];
        }
        float f = 0.0f;
#pragma unroll
        for (int t = 0; t < TILES; ++t) {
          f32x16 p = {};
          p = __builtin_amdgcn_mfma_f32_32x32x16_f16(ah[w][t], bl, p, 0, 0, 0);
          p = __builtin_amdgcn_mfma_f32_32x32x16_f16(al[w][t], bh, p, 0, 0, 0);
          p = __builtin_amdgcn_mfma_f32_32x32x16_f16(ah[w][t], bh, p, 0, 0, 0);
#pragma unroll
          for (int q = 0; q < 2; ++q) {
            float s = wy[0] * p[8 * q];
#pragma unroll
            for (int v = 1; v < 8; ++v) s = __builtin_fmaf(wy[v], p[8 * q + v], s);
            f = __builtin_fmaf(wx[2 * t + q], s, f);
          }
        }
        f += __shfl_xor(f, 32, 64);
        if (half == hl) res[c] = f;
      }
    }
    if (idx < 0) continue;  // padding
    float v[NC];
#pragma unroll
    for (int c = 0; c < NC; ++c)
      v[c] = idx & kPlaceNaN ? NAN : static_cast<float>(static_cast<double>(res[c]) * oscale);
    if (NC > 1 && in_place) {  // uniform
      recs[static_cast<int64_t>(g) * kWavePts + lane] =
          make_float4(v[0], v[NC > 1 ? 1 : 0], v[NC > 1 ? 2 : 0], 0.0f);
      continue;
    }
#pragma unroll
    for (int c = 0; c < NC; ++c) out[c * out_ld + (idx & ~kPlaceNaN)] = v[c];
  }
}

template <int NC>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(NC == 1 ? 3 : 2)))
k_band_points(const BinParams* __restrict__ prm, const BandState* __restrict__ st,
              const _Float16* __restrict__ G, int64_t gl, const double* __restrict__ centre,
              const int* __restrict__ wave_cell, float4* recs, bool in_place,
              float* __restrict__ out, int64_t out_ld) {
  __shared__ __attribute__((aligned(16))) char rows[4 * kWavePts * kRowMax];
  const int tiles = prm->band;
  if (tiles == kWinTiles[0])
    points_run<NC, kWinTiles[0], false>(rows, prm, st, G, gl, centre, wave_cell, recs, in_place,
                                        out, out_ld);
  else if (tiles == kWinTiles[1])
    points_run<NC, kWinTiles[1], (NC > 1)>(rows, prm, st, G, gl, centre, wave_cell, recs,
                                           in_place, out, out_ld);
  else if (tiles == kWinTiles[2])
    points_run<NC, kWinTiles[2], (NC > 1)>(rows, prm, st, G, gl, centre, wave_cell, recs,
                                           in_place, out, out_ld);
}

// Vector results from the record slots to the points' places (slot given), and
// the rest modes' part.  Random 16-byte reads, where writing the three
// components at random takes 130 us per 4e6 points more than writing them in
// order does, this 75 us.
constexpr int kGatherPts = 4;  // points per lane, 256 apart
__global__ void __launch_bounds__(256)
k_band_gather(const BinParams* __restrict__ prm, const BandReal* __restrict__ dr,
              const BandState* __restrict__ st, const float4* __restrict__ recs,
              const int* __restrict__ slot, const double* __restrict__ pos, int64_t ld, int64_t N,
              float* __restrict__ out, int64_t out_ld) {
  if (!prm->band) return;
  const int64_t p0 = static_cast<int64_t>(blockIdx.x) * (256 * kGatherPts) + threadIdx.x;
  float4 v[kGatherPts];
#pragma unroll
  for (int u = 0; u < kGatherPts; ++u) {
    const int64_t p = min(p0 + 256 * u, N - 1);
    v[u] = slot ? recs[slot[p]] : make_float4(out[p], out[out_ld + p], out[2 * out_ld + p], 0.0f);
  }
  const int n_rest = st->n_rest;
  if (n_rest > 0) {
    const auto rest = const_ptr(dr->rest);
    const double scale = dr->scale;
#pragma unroll
    for (int u = 0; u < kGatherPts; ++u) {
      const int64_t p = min(p0 + 256 * u, N - 1);
      const double x[3] = {pos[p], pos[ld + p], pos[2 * ld + p]};
      double t[3];
      sum_modes_vec<3>(rest, n_rest, x, t);
      v[u].x = static_cast<float>(static_cast<double>(v[u].x) + t[0] * scale);
      v[u].y = static_cast<float>(static_cast<double>(v[u].y) + t[1] * scale);
      v[u].z = static_cast<float>(static_cast<double>(v[u].z) + t[2] * scale);
    }
  }
#pragma unroll
  for (int u = 0; u < kGatherPts; ++u) {
    const int64_t p = p0 + 256 * u;
    if (p >= N) return;
    out[p] = v[u].x;
    out[out_ld + p] = v[u].y;
    out[2 * out_ld + p] = v[u].z;
  }
}

}  // namespace

BandPoints place_band_points(int64_t M, int64_t N, const ModeRec* modes, bool vec, double scale,
                             int64_t max_cells, int64_t all_cells, const double* box, void* state,
                             void* space, size_t bytes) {
  BandPoints b{};
  char* base = static_cast<char*>(space);
  size_t off = 0;
  auto take = [&](size_t n) {
    const size_t o = off;
    off += (n + 255) & ~static_cast<size_t>(255);
    return base + o;
  };
  // (256 bytes each at least, in a region of record groups)
  constexpr auto up = [](size_t n) { return (n + 255) & ~static_cast<size_t>(255); };
  char* st = static_cast<char*>(state);
  BinParams* prm = reinterpret_cast<BinParams*>(st);
  b.d = reinterpret_cast<BandReal*>(st + up(sizeof(BinParams)));
  b.st = reinterpret_cast<BandState*>(st + up(sizeof(BinParams)) + up(sizeof(BandReal)));
  BandReal& r = b.real;
  r.rest = reinterpret_cast<ModeRec*>(take(sizeof(ModeRec) * static_cast<size_t>(M)));
  r.bm = reinterpret_cast<BandMode*>(take(sizeof(BandMode) * static_cast<size_t>(M + kNodeModes)));
  // vector fields: the points' record slots, where most of the space is left
  const size_t slots = vec ? sizeof(int) * static_cast<size_t>(N) : 0;
  if (slots > 0 && 4 * slots < bytes) b.slot = reinterpret_cast<int*>(take(slots));
  if (off + (size_t(1) << 20) > bytes) return b;  // (a 45^3 of nodes and more)
  // half for the parts G, the rest for the sums F of the splits.  Whole kilobytes:
  // the low parts' windows are then as aligned as the high ones' (whole words)
  const size_t left = std::min<size_t>((bytes - off) / 2 / sizeof(float), size_t(1) << 28) &
                      ~static_cast<size_t>(255);
  b.G = take(left * sizeof(float));
  b.gl = static_cast<int64_t>(left);
  r.F = reinterpret_cast<float*>(base + off);
  r.fcap = std::min<int64_t>(static_cast<int64_t>((bytes - off) / sizeof(float)), b.gl);
  r.dim = 3;
  r.ncomp = vec ? 3 : 1;
  r.M = static_cast<int>(M);
  r.modes = modes;
  r.scale = scale;
  for (int d = 0; d < 3; ++d) r.cap[d] = 4096;
  b.args = PointsArgs{box, N, max_cells, all_cells, vec ? 1 : 0, prm};
  return b;
}

hipError_t launch_band_points(const BandPoints& b, bool vec, const double* centre,
                              const int* wave_cell, float4* recs, const double* pos,
                              int64_t pos_ld, float* out, int64_t out_ld, hipStream_t s) {
  BandLaunch L{};
  L.count = 1;
  L.dim = 3;
  L.d = b.d;
  L.st = b.st;
  const hipError_t e = launch_band_nodes(L, s);
  if (e != hipSuccess) return e;
  _Float16* G = static_cast<_Float16*>(b.G);
  k_band_sum<<<512, 256, 0, s>>>(b.d, b.st, G, b.gl);
  if (vec)
    k_band_points<3><<<2048, 256, 0, s>>>(b.args.prm, b.st, G, b.gl, centre, wave_cell, recs,
                                          b.slot != nullptr, out, out_ld);
  else
    k_band_points<1><<<2048, 256, 0, s>>>(b.args.prm, b.st, G, b.gl, centre, wave_cell, recs,
                                          b.slot != nullptr, out, out_ld);
  if (vec) {
    const int64_t per = 256 * kGatherPts;
    k_band_gather<<<static_cast<unsigned>((b.args.N + per - 1) / per), 256, 0, s>>>(
        b.args.prm, b.d, b.st, recs, b.slot, pos, pos_ld, b.args.N, out, out_ld);
  }
  return hipGetLastError();
}

}  // namespace gsc
