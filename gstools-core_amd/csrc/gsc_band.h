// Band-limited path of structured grids (band.hip): host-side plan and
// launcher.
#pragma once

#include <hip/hip_runtime.h>

#include "gsc_factored.h"
#include "gsc_internal.h"

#include <cmath>
#include <cstddef>
#include <cstdint>

namespace gsc {

constexpr int kFirstRunShared = 64;  // longest run of first-axis coordinates per work item

// A mode of the band: kap per axis place (see BandReal), theta, amplitude over
// phihat on every axis, projector per component.
struct alignas(16) BandMode {
  double kap[3];
  double th;
  float amp;
  float proj[3];
};

// One grid as the kernels of band.hip see it.  Axes in C order; a 2-D grid
// has its two axes in places 0 and 2 (len[1] = 1).
struct BandReal {
  const double* ax[3];
  int64_t len[3];
  int dim;
  int ncomp;             // field components: 1, or dim (incompressible)
  int M;
  int shared;            // one of many grids that run together (an ensemble): their
                         // first_run (at most kFirstRunShared); 0: alone
  int k_grid;            // the modes are a k-grid's (Fourier method): many at the band's faces
  int64_t gemm_tiles;    // block tiles of the factored GEMM on this grid
  const ModeRec* modes;  // the full mode table (KIND_SCALAR or KIND_FOURIER amplitudes)
  int cap[3];            // most nodes per axis the workspace holds
  int64_t fcap;          // values of F
  // workspace
  ModeRec* rest;         // M: the modes left to the factored GEMM, in order
  BandMode* bm;          // M + 16: the band's modes
  int* i0[3];            // len[d]: first node of a coordinate's window
  float* wt[3];          // axes 0 and 1: window weights, 8 per coordinate
  double* wt2;           // axis 2: 8 x len[2] window weights, node-major
  float* F;              // node values, a set per split
  float* t1;             // after the last axis
  float* t2;             // 3-D: after the middle axis
  float* out;
  double scale;
};

// What the plan kernel decides for a grid.
struct BandState {
  int n_in;    // modes in the band (0: the path is off, the GEMM takes all)
  int n_rest;  // modes left to the factored GEMM (padded sizes follow from it)
  int n[3];    // nodes per axis
  int ident[3];  // the axis' nodes are its own coordinates
  int splits;  // mode splits of the node sums
  int big;     // 128 x 128 node tiles
  int vec, first_cols, first_run;  // first axis' kernel: 16-byte accesses, columns per lane, run
  int last_rows;     // node lines per work item of the last axis' kernel
  int64_t items[4];  // work items: nodes, last, middle and first axis
  int amp_exp;       // amplitudes times 2^amp_exp in the node sums
  double out_scale;  // and their results times this
  double g_scale;  // point lists: node sums times this in the fp16 parts (out_scale has its inverse)
  double lo[3], h[3];  // node i at lo + i h
};

// Point lists (3-D, band_points.hip).
struct BinParams;
struct PointsArgs {
  const double* box;   // kBoxBlocks partial bounding boxes
  int64_t N;
  int64_t max_cells, all_cells;  // of the band path, of the local kernel
  int vec;             // the modes carry their component amplitudes (KIND_INCOMPR)
  BinParams* prm;      // cells of the band path; prm->band: whether it is taken
};
struct BandPoints {
  BandReal real;       // stored to *d by the planning kernel
  PointsArgs args;     // args.prm null: no space for the path
  BandReal* d;
  BandState* st;
  void* G;             // node values in fp16: high parts, from gl on the low parts
  int64_t gl;
  int* slot;           // null, or the points' record slots, which the sort leaves there (vector
                       // fields: results go to the slots first, then to the points' places)
};
// Whether the path is planned: where the local kernel's time per point, 1e-13 s
// a mode (1.75e-13 s for three components), exceeds the interpolation's, that of
// 250 (450) modes, by what the path's launches and nodes cost (about 20 us), and
// from kBandPoints points on: below, the local kernel splits a record group's rough
// modes over waves, which no band's rest modes get back (32000 points of 6624
// exponential modes, 500^3, l = 20: 172 us, 1080 us with their band).  A plan that
// takes no mode costs 4 to 10 us.  Measured on one MI355X, 500^3 and l = 20: 2.6e5
// points of 1000 modes 107 us either way, 5e5 128 us without the path and 98 us with
// it; 3e6 of 300 modes 298 us without, 310 us planned and not taken.
constexpr int64_t kBandPoints = 65536;
inline bool band_points_pay(int64_t M, int64_t N, bool vec) {
  return N >= kBandPoints &&
         static_cast<double>(N) * static_cast<double>(M - (vec ? 450 : 250)) >= 2e8;
}
BandPoints place_band_points(int64_t M, int64_t N, const ModeRec* modes, bool vec, double scale,
                             int64_t max_cells, int64_t all_cells, const double* box, void* state, void* space, size_t bytes);
// After the cell sort (over args.prm's cells where prm->band): the node values
// and the interpolation; nothing where the plan left the band empty.
hipError_t launch_band_points(const BandPoints& b, bool vec, const double* centre,
                              const int* wave_cell, float4* recs, const double* pos,
                              int64_t pos_ld, float* out, int64_t out_ld, hipStream_t s);

// Seconds of a factored GEMM of m modes in `tiles` block tiles, measured on one
// MI355X (256 CUs): a 16-mode chunk of a 256 x 128 tile takes a CU 1.45 us, 1.1 us
// where none has a second tile.  shared: a grid's share of many grids' launches.
__host__ __device__ inline float factored_seconds(int64_t tiles, int m, bool shared) {
  if (m <= 0) return 0.0f;
  const float rounds = static_cast<float>(tiles) / 256.0f;
  const float chunks = static_cast<float>(2 * ((m + 31) / 32));
  if (shared) return rounds * chunks * 1.45e-6f + 6e-6f;
  return (rounds <= 1.0f ? 1.1e-6f : ceilf(rounds) * 1.45e-6f) * chunks + 5e-6f;
}
// Whether the band is planned for one grid.  Where the plan takes no mode (or few
// of a heavy-tailed spectrum), its kernel and those that find nothing to do cost
// 20 us, which grids of shorter GEMMs may not get back: with it planned from 50 us
// on, 247 x 795 x 2 values of 868 exponential modes took 108 us instead of 82 and 719 x
// 229 of 1181 121 instead of 96, though 419 x 1670 of 943 Gaussian ones 43 instead of
// 84.  Above, 71 x 287 x 24 x 3 values of 804 exponential modes take 136 us (121 without),
// 197 x 699 x 2 of 1396 71 (115).
inline bool band_grid_pays(int64_t tiles, int64_t M) {
  return factored_seconds(tiles, static_cast<int>(M), false) >= 100e-6f;
}

// Workspace of one grid: bytes of everything behind `off` fields below, and
// the placement (offsets from a 256-byte aligned base).  on = false where the
// path is never taken for the sizes.
struct BandPlan {
  bool on;
  int cap[3];
  int64_t fcap;
  int64_t len[3];
  int ncomp;
  size_t rest, bm, i0[3], wt[3], F, t1, t2, bytes;
};
BandPlan plan_band(int dim, int64_t M, const int64_t* shape, int ncomp);

// Fills the geometry and workspace pointers of a BandReal from its plan.
void band_place(const BandPlan& p, void* base, BandReal* r);

// The grids of a launch (device arrays).
constexpr int kBandLists = 4;
struct BandLaunch {
  int count, dim;
  BandReal* d;
  BandState* st;
  int64_t* pre;   // many grids: kBandLists x (count + 1); one: null
  int* any_rest;  // null, or a counter (zero before) of the grids with rest modes
};

// Whether the band path pays in an ensemble, by the plans of its realisations (r and
// st on the host, `count` of them): its launches against what it takes off the
// factored part, in `gemms` GEMM launches, which is shared with the realisations
// without a plan (other).
struct EnsChunks {  // chunks of 16 modes
  double tiles = 0.0, tables = 0.0;  // of all block tiles, of all realisations
  int longest = 0;                   // of one
  void add(int64_t n, int chunks) {
    tiles += static_cast<double>(n) * chunks;
    tables += chunks;
    if (chunks > longest) longest = chunks;
  }
};
bool band_ensemble_pays(const BandReal* r, const BandState* st, int count, int gemms,
                        const EnsChunks& other);

// The path's kernels: the plan, the node values and, when `rest` is given (one
// grid), the factored tables of the rest modes in blocks of the same launch;
// then, after the factored GEMM of the rest modes (st[i].n_rest of d[i].rest)
// has written its part of every output, band_finish adds (or, without rest
// modes, writes) the band's part.  one: a single grid's description, which the
// plan kernel then stores to d[0]; null where d holds them.
hipError_t launch_band_plan(const BandLaunch& L, const BandReal* one, const TableArgs* rest,
                            hipStream_t s);
hipError_t launch_band_finish(const BandLaunch& L, hipStream_t s);
// The plans alone.
hipError_t launch_band_plans(const BandLaunch& L, hipStream_t s);
// The node values alone, for one grid planned elsewhere (point lists).
hipError_t launch_band_nodes(const BandLaunch& L, hipStream_t s);

}  // namespace gsc
