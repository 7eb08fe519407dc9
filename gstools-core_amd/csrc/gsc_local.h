// Spatial cells of the point-list kernels (direct_local.hip, band_points.hip).
#pragma once

#include <hip/hip_runtime.h>

#include "gsc_internal.h"

#include <cstdint>

namespace gsc {

constexpr int kWavePts = 64;      // point slots per record group (one wave)
constexpr int kBoxBlocks = 1024;  // partial bounding boxes
constexpr int kBandStateGroups = 4;  // record groups that hold the band path's state
constexpr int kMaxCells = 16384;  // cell counters of one block fill 64 KB of LDS

struct alignas(16) BinParams {
  double lo[3];
  double h[3];
  double inv_h[3];
  double inv_f[3];  // 1 / f
  int n[3];       // cells per dimension
  int f[3];       // cells per coarse cell and dimension
  int C[3];       // coarse cells per dimension
  int F;          // f0 f1 f2
  int ncoarse;    // C0 C1 C2
  int ncells;     // ncoarse F: cell numbers (coarse-major, some empty past n)
  int nwaves;
  int n_smooth;
  int n_rough;
  int band;       // 0, or the tiles per window of the band path (band_points.hip)
  // its nodes: node0 + i / inv_node, i < nodes
  int nodes[3];
  double node0[3], inv_node[3];
};

// Records of the band path's points (see scatter_point).
constexpr double kPlaceUnit = 268435456.0;  // 2^28
constexpr uint32_t kPlaceMask = (1u << 28) - 1;
constexpr int kPlaceNaN = 1 << 30;  // (point indices are below)

// The cell grid of n cells per dimension over [lo, lo + ext]: coarse cells of
// f_k cells per dimension, at most 8 per dimension; the numbering covers
// whole coarse cells, so it may exceed n0 n1 n2; n shrinks until it stays
// within max_cells.  Fills every field but the counts.
__device__ inline void cell_grid(int (&n)[3], const double (&lo)[3], const double (&ext)[3],
                                 int64_t max_cells, BinParams& P) {
  int f[3], C[3];
  for (;;) {
    int64_t total = 1;
    for (int k = 0; k < 3; ++k) {
      f[k] = (n[k] + 7) / 8;
      C[k] = (n[k] + f[k] - 1) / f[k];
      total *= static_cast<int64_t>(f[k]) * C[k];
    }
    if (total <= max_cells) break;
    for (int k = 0; k < 3; ++k) n[k] = n[k] > 1 ? n[k] * 4 / 5 : 1;
  }
  P = BinParams{};
  for (int k = 0; k < 3; ++k) {
    P.lo[k] = lo[k];
    P.n[k] = n[k];
    P.f[k] = f[k];
    P.C[k] = C[k];
    // a dimension without extent (a planar slice) gets width 0: every
    // point sits at the cell centre there (xi = 0) and the dimension adds
    // nothing to a mode's local-phase bound (half_cell_exp(0) scales by 1)
    P.h[k] = ext[k] > 0.0 ? ext[k] / n[k] : 0.0;
    P.inv_h[k] = ext[k] > 0.0 ? 1.0 / P.h[k] : 0.0;
    P.inv_f[k] = 1.0 / f[k];
  }
  P.F = f[0] * f[1] * f[2];
  P.ncoarse = C[0] * C[1] * C[2];
  P.ncells = P.ncoarse * P.F;
}

// Band path: first node, on axis d, of the window of the cell centred at X.  A
// point's own window starts at node ceil(u - 4), u its place in nodes, and the
// points reach half a cell (+ rounding) from the centre; even on the last axis.
__device__ __forceinline__ int window_base(const BinParams& P, int d, double X) {
  const double u = (X - P.node0[d]) * P.inv_node[d];
  const int b = static_cast<int>(ceil(u - 0.5 * P.h[d] * P.inv_node[d] - 1e-6)) - 4;
  const int win = d == 0 ? 2 * P.band : 16;
  return min(max(d == 2 ? b & ~1 : b, 0), P.nodes[d] - win);
}

// Centre of cell number e (FP64).
template <int D>
__device__ __forceinline__ void cell_centre(const BinParams& P, int e, double (&X)[3]) {
  X[0] = X[1] = X[2] = 0.0;
  int cc = e / P.F, l = e - (e / P.F) * P.F;
#pragma unroll
  for (int k = D - 1; k >= 0; --k) {
    const int ck = cc % P.C[k], lk = l % P.f[k];
    cc /= P.C[k];
    l /= P.f[k];
    X[k] = P.lo[k] + (ck * P.f[k] + lk + 0.5) * P.h[k];
  }
}

}  // namespace gsc
