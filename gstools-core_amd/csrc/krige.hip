// Kriging calculators (src/krige.rs:24-118): with n conditions and N targets,
//   krig_fac_i(j) = sum_k mat[k][i] vecs[k][j]        (W = mat^T vecs)
//   field[j]      = sum_i cond[i] krig_fac_i(j)
//   error[j]      = sum_i vecs[i][j] krig_fac_i(j)
// (krige.rs:47-57: `m_row` walks the columns of krig_mat).
//
// field and error (calculator_field_krige_and_variance): the error is the
// quadratic form v^T mat v of a target's column v, which only sees the
// symmetric part of mat, so it is summed over the lower triangle alone:
//   error[j] = sum_i v_i T_i,  T_i = sum_{k <= i} S_ik v_k,
//   S_ii = mat_ii,  S_ik = mat_ik + mat_ki (k < i),
// n^2 N flops instead of 2 n^2 N, and the field takes the form below.  T is
// computed tile by tile on the FP64 matrix cores (v_mfma_f64_16x16x4f64) and
// contracted with vecs in the tile epilogue, so it never reaches memory.
// The T_i are larger than the full row sums (mat v cancels, half of it does
// not), and K passes half as many of them, so their rounding errors would be 1.4 times
// the full form's.  So T is summed in segments of about n / 3 conditions (64 at
// least), each contracted by itself, eight rows at a time, and the sums of those carry
// their rounding errors along (two-sum, s + c).  Against extended precision, the rms
// relative error of error[j] for an exponential covariance is 1.46e-14 at n = 1000 and
// 4.6e-15 at 385, 1.86e-14 and 5.6e-15 in the full form (segments of n / 4: 1.0e-14 and
// 4.4e-15, 5 % more time; one segment: 2.5e-14 and 7.9e-15, 3 to 8 % less).
// A block owns 128 rows i (four waves of two 16-row MFMA tiles, so every B
// operand read from LDS feeds two matrix instructions) and 128 targets j (eight
// 16-column MFMA tiles per wave); K runs over the conditions up to the block's last
// row in LDS-staged chunks of 16 (the accumulators, 128 registers, and the next
// chunk's prefetch fit two waves per SIMD).  Bound by the FP64 matrix cores: n =
// 1000, N = 1e6 takes 20.2 ms against 36.0 ms for the full form (56 TFLOP/s executed,
// the diagonal blocks' upper halves included).  Splits of the row blocks write their
// partial sums, which a second kernel adds in a fixed order (results are
// bitwise reproducible).  Few targets take the full form, W = mat^T vecs with
// one block per row block (see launch_krige).
//
// field: the sum reassociated as field[j] = sum_k vecs[k][j] w[k],
// w = mat cond (n^2 + 2 n N flops).  The reassociation changes rounding only, of
// finite fields.  With the error, the others are summed again as written above;
// alone (calculator_field_krige) an infinite entry of cond makes every w infinite, so
// its fields are NaN.  Alone it is bound by reading vecs once.
#include "gsc_device.h"
#include "gsc_internal.h"

#include <hip/hip_runtime.h>

#include <algorithm>

namespace gsc {
namespace {

typedef double f64x4 __attribute__((ext_vector_type(4)));

constexpr int kRS = 2;        // 16-row MFMA tiles per wave
constexpr int kKI = 64 * kRS; // rows i per block (four waves of 16 kRS)
constexpr int kKK = 16;       // conditions k per LDS chunk
constexpr int kTJ = 8;   // 16-column MFMA tiles per wave: kKJ = 16 kTJ targets per block
constexpr int kKJ = 16 * kTJ;
constexpr int64_t kSlots = 512;       // resident blocks: two per CU
constexpr int64_t kTriBlocks = 3 * kSlots;  // blocks wanted of the triangle form
constexpr double kSymCost = 45.0;     // the triangle's launch, in conditions of a round (0.3 us)
constexpr double kTriSure = 0.95;     // of the full form's time, which has to be beaten
constexpr int kXcds = 8; // blocks are dispatched to the XCDs round-robin

// Block b -> (split q of nq, target block jb): the splits of one target
// block run on one XCD, so its columns of vecs stay in that XCD's L2.
__device__ __forceinline__ bool krige_block(int nq, int njb, int& q, int& jb) {
  const int b = blockIdx.x;
  const int xcd = b % kXcds, s = b / kXcds;
  jb = xcd + kXcds * (s / nq);
  q = s % nq;
  return jb < njb;
}

// s + c += v exactly to second order (two-sum).
__device__ __forceinline__ void two_sum(double v, double& s, double& c) {
  const double t = s + v, z = t - s;
  c += (s - (t - z)) + (v - z);
  s = t;
}

// s + c += a b, the product with its rounding error.
__device__ __forceinline__ void two_prod_sum(double a, double b, double& s, double& c) {
  const double p = a * b;
  c += __builtin_fma(a, b, -p);
  two_sum(p, s, c);
}

// s + c; infinities turn the carried rounding error into NaN: the plain sum then.
__device__ __forceinline__ double with_carry(double s, double c) {
  return isfinite(c) ? s + c : s;
}

// w[k] = sum_i mat[k][i] cond[i]: one wave per row k, lanes over i, then a
// fixed-order tree over the lanes.  CARRY: with the rounding errors.
template <bool CARRY>
__device__ __forceinline__ void krige_w_row(int64_t n, int64_t k, const double* __restrict__ mat,
                                            const double* __restrict__ cond,
                                            double* __restrict__ w) {
  const int lane = threadIdx.x & 63;
  if (k >= n) return;
  double s = 0.0, c = 0.0;
  for (int64_t i = lane; i < n; i += 64) {
    if constexpr (CARRY) two_prod_sum(mat[k * n + i], cond[i], s, c);
    else s = __builtin_fma(mat[k * n + i], cond[i], s);
  }
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) {
    if constexpr (CARRY) {
      const double s2 = __shfl_xor(s, off, 64), c2 = __shfl_xor(c, off, 64);
      c += c2;
      two_sum(s2, s, c);
    } else {
      s += __shfl_xor(s, off, 64);
    }
  }
  if (lane == 0) w[k] = CARRY ? with_carry(s, c) : s;
}

// The triangle in k-major order, st[k][i] = S_ik for k <= i < n and zero
// elsewhere, in ld rows of ld = round_up(n, 16) (blocks [0, tiles): 32 x 32
// tiles, the mirrored tile transposed through LDS), and w (the blocks after
// them).
constexpr int kSymTile = 32;
__global__ void __launch_bounds__(256)
k_krige_sym(int64_t n, int64_t ld, int64_t nt, const double* __restrict__ mat,
            const double* __restrict__ cond, double* __restrict__ st, double* __restrict__ w) {
  __shared__ double tr[kSymTile][kSymTile + 1];
  const int64_t b = blockIdx.x;
  if (b >= nt * nt) {  // uniform over the block
    krige_w_row<true>(n, (b - nt * nt) * 4 + (threadIdx.x >> 6), mat, cond, w);
    return;
  }
  const int64_t k0 = b / nt * kSymTile, i0 = b % nt * kSymTile;
  const int tx = threadIdx.x % kSymTile, ty = threadIdx.x / kSymTile;
  const bool upper = k0 <= i0;
  if (upper) {  // uniform over the block
#pragma unroll
    for (int u = 0; u < kSymTile; u += 8) {
      const int64_t i = i0 + ty + u, k = k0 + tx;
      tr[tx][ty + u] = i < n && k < n ? mat[i * n + k] : 0.0;
    }
    __syncthreads();
  }
#pragma unroll
  for (int u = 0; u < kSymTile; u += 8) {
    const int64_t k = k0 + ty + u, i = i0 + tx;
    double v = 0.0;
    if (upper && k <= i && i < n) v = k == i ? mat[k * n + i] : mat[k * n + i] + tr[ty + u][tx];
    if (k < ld && i < ld) st[k * ld + i] = v;
  }
}

// LDS of a block: the staged chunk of mat (kKK x kKI) and vecs (kKK x kKJ), and the
// epilogue's partial sums (2 x 16 x kKJ): their place is the chunk's after the K loop,
// or their own in the triangle form, which adds to them between segments of K.
struct KrigeStage {
  double m[kKK][kKI + 1];
  double v[kKK][kKJ + 1];
};
struct KrigeRed {
  double r0[16][kKJ + 1];
  double r1[16][kKJ + 1];
};
template <bool TRI>
struct KrigeSmem {
  union {
    KrigeStage st;
    KrigeRed red;
  };
};
template <>
struct KrigeSmem<true> {
  KrigeStage st;
  KrigeRed red;
};

// MFMA operand / result layouts (v_mfma_f64_16x16x4f64, verified on gfx950):
//   A: lane l holds A[l % 16][l / 16], B: lane l holds B[l / 16][l % 16],
//   D: lane l, item it holds D[4 it + l / 16][l % 16].
// Here A[i][k] = mat[k][i] (16 rows i of one of the wave's kRS tiles), B[k][j] = vecs[k][j].
// Every row block reads its part of mat once per kKJ targets, so the target
// width sets mat's share of the traffic (n^2 8 / kKJ bytes per target, half
// of that in the triangle form).
//
// TRI, the triangle form: mat is the triangle st (ld rows of ld), cw is w.
// Split q of nq takes the row blocks q, 2 nq - 1 - q, 2 nq + q, .. (about
// equal triangle parts) one after the other and keeps the error sums (s, c)
// of its columns; with one split they are final, else they go to part rows
// 2 q and 2 q + 1.  K runs in segments of seg conditions, each contracted with the
// block's vecs by itself.  The last row block, whose K loop
// passes every condition, gives the field (the staged vecs times w).
// FULL, W = mat^T vecs in full: cw is cond, split q is row block q, seg is at
// least n, and the partial sums of field and error go to part rows q and nq + q.
// REDO, after the triangle form: the full form (one split) of the targets whose field or
// error is not finite there.  Infinities spread differently in it (the triangle's zeros
// and w), and S_ik may overflow where mat does not; such targets' results are those
// of the full form, whatever the number of targets.  Blocks without any end at once
// (N = 1e6: 22 us).
// SKIP: waves whose rows all lie past the last condition (or, TRI, past the chunk)
// leave out the matrix instructions.  Not in FULL from kKI / 2 conditions on: the branch
// costs more than the idle rows do (n = 298, N = 28766: 144 us without it, 168 with;
// 568 and 31472: 409 and 460; 32 and 1e6: 245 and 222).
enum Form { FULL, TRIANGLE, REDO };
template <Form FORM, bool SKIP = FORM != FULL>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2, 2)))
k_krige_tiles(int64_t n, int64_t N, const double* __restrict__ mat, int64_t ld,
              const double* __restrict__ vecs, int64_t vld, const double* __restrict__ cw,
              int nib, int nq, int njb, int seg, double* __restrict__ part,
              double* __restrict__ field, double* __restrict__ error) {
  constexpr bool TRI = FORM == TRIANGLE;
  __shared__ KrigeSmem<TRI> sm;
  int q, jb;
  if (!krige_block(nq, njb, q, jb)) return;
  const int64_t j0 = static_cast<int64_t>(jb) * kKJ;
  bool redo = false;
  double f_all = 0.0, e_all = 0.0;  // REDO: sums over the row blocks
  if constexpr (FORM == REDO) {
    const int64_t j = j0 + threadIdx.x;
    if (threadIdx.x < kKJ && j < N) redo = !isfinite(field[j]) || !isfinite(error[j]);
    if (!__syncthreads_or(redo)) return;
  }
  const int lane = threadIdx.x & 63, g = lane >> 4, jl = lane & 15;
  const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  // this thread's share of a chunk: mat[k0 + tm_k + kStepM u][i0 + tm_i] and
  // vecs[k0 + tv_k + kStepV u][j0 + tv_j] (zero outside), i.e. element
  // e = threadIdx.x + 256 u of the row-major chunk tiles
  constexpr int kPerM = kKK * kKI / 256, kPerV = kKK * kKJ / 256;
  constexpr int kStepM = 256 / kKI, kStepV = 256 / kKJ;
  const int tm_k = threadIdx.x / kKI, tm_i = threadIdx.x % kKI;
  const int tv_k = threadIdx.x / kKJ, tv_j = threadIdx.x % kKJ;
  const int n32 = static_cast<int>(n);  // n <= 2^24
  const int64_t m_step = kStepM * ld, v_step = kStepV * vld;
  if constexpr (TRI) {  // the lane's own slots of the error sums (s, c)
#pragma unroll
    for (int t = 0; t < kTJ; ++t) {
      sm.red.r0[4 * wv + g][16 * t + jl] = 0.0;
      sm.red.r1[4 * wv + g][16 * t + jl] = 0.0;
    }
  }
  for (int turn = 0;; ++turn) {
    const int ib = turn * nq + (turn & 1 ? nq - 1 - q : q);
    if (turn * nq >= nib) break;
    if (ib >= nib) continue;
    const int64_t i0 = static_cast<int64_t>(ib) * kKI;
    // the wave's rows start at row0 of the block (kRS tiles)
    const int row0 = 16 * kRS * wv;
    // K ends with the last condition; in the triangle form with the block's
    // last row, and the wave needs the chunks up to its own rows only
    const int kend = static_cast<int>(TRI ? min(i0 + kKI, n) : n);
    const int kw = static_cast<int>(i0 + row0 < n ? (TRI ? min(i0 + row0 + 16 * kRS, n) : n) : 0);
    const bool with_field = TRI && ib == nib - 1;
    double rm[kPerM], rv[kPerV];
    double fs = 0.0, fc = 0.0;  // this thread's part of field[j0 + tv_j]
    const double* mp = mat + min(i0 + tm_i, n - 1) + static_cast<int64_t>(tm_k) * ld;
    const double* vp = vecs + min(j0 + tv_j, N - 1) + static_cast<int64_t>(tv_k) * vld;
    // rows past n read row 0 and carry zeros; columns past n (mat) and N
    // (vecs) read the last one, and what they give is not used
    auto gload = [&](int k0) {
      if (FORM == FULL && k0 + kKK <= n32) {  // uniform: no row past the last condition
        const double* pm = mp + static_cast<int64_t>(k0) * ld;
        const double* pv = vp + static_cast<int64_t>(k0) * vld;
#pragma unroll
        for (int u = 0; u < kPerM; ++u) rm[u] = pm[u * m_step];
#pragma unroll
        for (int u = 0; u < kPerV; ++u) rv[u] = pv[u * v_step];
        return;
      }
      const double* pm = mat + (TRI ? i0 + tm_i : min(i0 + tm_i, n - 1));
      const double* pv = vecs + min(j0 + tv_j, N - 1);
      // opaque: the rows' addresses are formed here, not kept over the turns
      // (they would take the registers of the prefetch)
      __asm__ volatile("" : "+v"(pm), "+v"(pv));
      const double* qm = pm + static_cast<int64_t>(tm_k + k0) * ld;
      const double* qv = pv + static_cast<int64_t>(tv_k + k0) * vld;
#pragma unroll
      for (int u = 0; u < kPerM; ++u)
        rm[u] = *(TRI || k0 + tm_k + kStepM * u < n32 ? qm + u * m_step : pm);
#pragma unroll
      for (int u = 0; u < kPerV; ++u)
        rv[u] = *(k0 + tv_k + kStepV * u < n32 ? qv + u * v_step : pv);
    };
    gload(0);
    for (int s0 = 0; s0 < kend; s0 += seg) {
      const int s1 = min(s0 + seg, kend);
      f64x4 acc[kRS][kTJ];
#pragma unroll
      for (int r = 0; r < kRS; ++r)
#pragma unroll
        for (int t = 0; t < kTJ; ++t) acc[r][t] = f64x4{0.0, 0.0, 0.0, 0.0};
      for (int k0 = s0; k0 < s1; k0 += kKK) {
        if (k0 + kKK > n32) {  // uniform: the chunk past the last condition
#pragma unroll
          for (int u = 0; u < kPerM; ++u)
            if (k0 + tm_k + kStepM * u >= n32) rm[u] = 0.0;
#pragma unroll
          for (int u = 0; u < kPerV; ++u)
            if (k0 + tv_k + kStepV * u >= n32) rv[u] = 0.0;
        }
#pragma unroll
        for (int u = 0; u < kPerM; ++u) sm.st.m[tm_k + kStepM * u][tm_i] = rm[u];
#pragma unroll
        for (int u = 0; u < kPerV; ++u) sm.st.v[tv_k + kStepV * u][tv_j] = rv[u];
        if (with_field) {  // uniform over the block
          double p = 0.0;
#pragma unroll
          for (int u = 0; u < kPerV; ++u)
            p = __builtin_fma(cw[min(k0 + tv_k + kStepV * u, n32 - 1)], rv[u], p);
          two_sum(p, fs, fc);
        }
        __syncthreads();
        // the next chunk's loads are in flight during this chunk's MFMAs
        if (k0 + kKK < kend) gload(k0 + kKK);
        __builtin_amdgcn_sched_barrier(0);
        if (!SKIP || k0 < kw) {  // uniform per wave
#pragma unroll
          for (int kk = 0; kk < kKK; kk += 4) {
            double a[kRS];
#pragma unroll
            for (int r = 0; r < kRS; ++r) a[r] = sm.st.m[kk + g][row0 + 16 * r + jl];
#pragma unroll
            for (int t = 0; t < kTJ; ++t) {
              const double b = sm.st.v[kk + g][16 * t + jl];
#pragma unroll
              for (int r = 0; r < kRS; ++r)
                acc[r][t] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[r], b, acc[r][t], 0, 0, 0);
            }
          }
        }
        __syncthreads();
      }
      if (TRI && s0 >= kw) continue;  // uniform per wave: none of the segment's sums
      // acc[r][t][it] = W, or the segment's part of T, [i0 + row0 + 16 r + 4 it + g][j0 + 16 t + jl];
      // between segments the next t's vecs are read while this one's are summed (8 loads
      // at a time: registers)
      double va[kRS][4], vb[kRS][4];
      auto vload = [&](int t, double (&v)[kRS][4]) {
        int64_t j = j0 + 16 * t + jl;
        __asm__ volatile("" : "+v"(j));  // addresses formed here, not kept over the K loop
        const double* p = vecs + min(j, N - 1);
#pragma unroll
        for (int r = 0; r < kRS; ++r)
#pragma unroll
          for (int it = 0; it < 4; ++it)
            v[r][it] = p[min(i0 + row0 + 16 * r + 4 * it + g, n - 1) * vld];
      };
      auto contract = [&](int t, const double (&v)[kRS][4]) {
        double p0 = 0.0, p1 = 0.0;  // TRI: of the error; else of field, error
#pragma unroll
        for (int r = 0; r < kRS; ++r)
#pragma unroll
          for (int it = 0; it < 4; ++it) {
            const int64_t i = i0 + row0 + 16 * r + 4 * it + g;
            const double vi = i < n ? v[r][it] : 0.0, tv = i < n ? acc[r][t][it] : 0.0;
            if constexpr (!TRI) p1 = __builtin_fma(vi, tv, p1);
            p0 = __builtin_fma(TRI ? vi : (i < n ? cw[i] : 0.0), tv, p0);
          }
        double& s = sm.red.r0[4 * wv + g][16 * t + jl];
        double& c = sm.red.r1[4 * wv + g][16 * t + jl];
        if constexpr (TRI) {
          double s0 = s, c0 = c;
          two_sum(p0, s0, c0);
          s = s0;
          c = c0;
        } else {
          s = p0;
          c = p1;
        }
      };
      if constexpr (TRI) {
        vload(0, va);
#pragma unroll
        for (int t = 0; t < kTJ; t += 2) {
          vload(t + 1, vb);
          __builtin_amdgcn_sched_barrier(0);
          contract(t, va);
          if (t + 2 < kTJ) vload(t + 2, va);
          __builtin_amdgcn_sched_barrier(0);
          contract(t + 1, vb);
        }
      } else {
#pragma unroll
        for (int t = 0; t < kTJ; ++t) {
          vload(t, va);
          contract(t, va);
          __builtin_amdgcn_sched_barrier(0);
        }
      }
    }
    if constexpr (!TRI) {
      __syncthreads();
      const int64_t j = j0 + threadIdx.x;
      if (threadIdx.x < kKJ && j < N) {
        double f = 0.0, e = 0.0;
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          f += sm.red.r0[r][threadIdx.x];
          e += sm.red.r1[r][threadIdx.x];
        }
        if constexpr (FORM == REDO) {
          f_all += f;
          e_all += e;
        } else {
          part[static_cast<int64_t>(q) * N + j] = f;
          part[static_cast<int64_t>(nq + q) * N + j] = e;
        }
      }
      if constexpr (FORM == FULL) break;
      __syncthreads();  // the sums are read
    } else if (with_field) {  // the kStepV threads of a column, through the stage
      sm.st.m[tv_k][tv_j] = fs;
      sm.st.v[tv_k][tv_j] = fc;
      __syncthreads();
      if (tv_k == 0 && j0 + tv_j < N) {
#pragma unroll
        for (int r = 1; r < kStepV; ++r) {
          fc += sm.st.v[r][tv_j];
          two_sum(sm.st.m[r][tv_j], fs, fc);
        }
        field[j0 + tv_j] = with_carry(fs, fc);
      }
      __syncthreads();
    }
  }
  if constexpr (FORM == REDO) {
    if (redo) {
      field[j0 + threadIdx.x] = f_all;
      error[j0 + threadIdx.x] = e_all;
    }
  }
  if constexpr (TRI) {
    __syncthreads();
    const int64_t j = j0 + threadIdx.x;
    if (threadIdx.x < kKJ && j < N) {
      double es = 0.0, ec = 0.0;
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        ec += sm.red.r1[r][threadIdx.x];
        two_sum(sm.red.r0[r][threadIdx.x], es, ec);
      }
      if (nq == 1) {
        error[j] = with_carry(es, ec);
      } else {
        part[static_cast<int64_t>(2 * q) * N + j] = es;
        part[static_cast<int64_t>(2 * q + 1) * N + j] = ec;
      }
    }
  }
}

// Adds the partial sums of nq splits (k_krige_tiles) in order.
template <bool TRI>
__global__ void __launch_bounds__(256)
k_krige_sum(int64_t N, int nq, const double* __restrict__ part, double* __restrict__ field,
            double* __restrict__ error) {
  const int64_t j = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
  if (j >= N) return;
  if constexpr (TRI) {
    double s = 0.0, c = 0.0;
    for (int q = 0; q < nq; ++q) {
      c += part[static_cast<int64_t>(2 * q + 1) * N + j];
      two_sum(part[static_cast<int64_t>(2 * q) * N + j], s, c);
    }
    error[j] = with_carry(s, c);
  } else {
    double f = 0.0, e = 0.0;
    for (int q = 0; q < nq; ++q) {
      f += part[static_cast<int64_t>(q) * N + j];
      e += part[static_cast<int64_t>(nq + q) * N + j];
    }
    field[j] = f;
    error[j] = e;
  }
}

__global__ void __launch_bounds__(256)
k_krige_w(int64_t n, const double* __restrict__ mat, const double* __restrict__ cond,
          double* __restrict__ w) {
  krige_w_row<false>(n, static_cast<int64_t>(blockIdx.x) * 4 + (threadIdx.x >> 6), mat, cond, w);
}

// field[j] = sum_k vecs[k][j] w[k]: one lane per target, rows in order;
// kFieldRows rows' loads are issued before their FMAs, so that many loads
// per wave are in flight.  WS > 1 (few targets): a block of WS waves shares 64
// targets, each a run of the rows, and adds the runs in order; one wave for all
// rows leaves most of the chip waiting for few loads (30011 targets, 137 rows:
// 8.9 us, 6.8 us with 8 waves).
constexpr int kFieldRows = 8;
constexpr int64_t kFieldSplit = 32768;
template <int WS>
__global__ void __launch_bounds__(WS > 1 ? 64 * WS : 256)
k_krige_field(int64_t n, int64_t N, const double* __restrict__ vecs, int64_t vld,
              const double* __restrict__ w, double* __restrict__ field) {
  __shared__ double part[WS > 1 ? WS : 1][64];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int64_t j = WS > 1 ? static_cast<int64_t>(blockIdx.x) * 64 + lane
                           : static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
  if (WS == 1 && j >= N) return;
  const double* p = vecs + (j < N ? j : N - 1);
  double f = 0.0;
  int64_t k = WS > 1 ? n * wave / WS : 0;
  const int64_t k1 = WS > 1 ? n * (wave + 1) / WS : n;
  for (; k + kFieldRows <= k1; k += kFieldRows) {
    double v[kFieldRows];
#pragma unroll
    for (int u = 0; u < kFieldRows; ++u) v[u] = p[(k + u) * vld];
#pragma unroll
    for (int u = 0; u < kFieldRows; ++u) f = __builtin_fma(v[u], w[k + u], f);
  }
  for (; k < k1; ++k) f = __builtin_fma(p[k * vld], w[k], f);
  if constexpr (WS > 1) {
    part[wave][lane] = f;
    __syncthreads();
    if (wave > 0 || j >= N) return;
#pragma unroll
    for (int q = 1; q < WS; ++q) f += part[q][lane];
  }
  field[j] = f;
}

}  // namespace

size_t krige_work_bytes(int64_t n, int64_t N, bool with_error) {
  if (!with_error) return sizeof(double) * static_cast<size_t>(n > 0 ? n : 1);
  const int64_t nib = (n + kKI - 1) / kKI;
  return 2 * sizeof(double) * static_cast<size_t>(nib > 0 ? nib : 1) *
         static_cast<size_t>(N > 0 ? N : 1);
}

hipError_t launch_krige(int64_t n, int64_t N, const double* mat, const double* vecs, int64_t vld,
                        const double* cond, double* field, double* error, void* work,
                        hipStream_t s) {
  if (N <= 0) return hipSuccess;
  const unsigned wb = static_cast<unsigned>((n + 3) / 4), jb = static_cast<unsigned>((N + 255) / 256);
  if (!error) {
    double* w = static_cast<double*>(work);
    if (n > 0) k_krige_w<<<wb, 256, 0, s>>>(n, mat, cond, w);
    // 8 waves per 64 targets while one per 64 leaves CUs with fewer than two
    // (n = 1000, us with one wave and with eight: 1000 targets 52.5 and 16.6, 30000
    // 88 and 52, 65536 98 and 117: rows read in eight places at a time)
    if (n >= 64 && N <= kFieldSplit)
      k_krige_field<8><<<static_cast<unsigned>((N + 63) / 64), 512, 0, s>>>(n, N, vecs, vld, w,
                                                                            field);
    else
      k_krige_field<1><<<jb, 256, 0, s>>>(n, N, vecs, vld, w, field);
    return hipGetLastError();
  }
  const int nib = static_cast<int>((n + kKI - 1) / kKI);
  const int64_t njb = (N + kKJ - 1) / kKJ;
  auto blocks = [njb](int64_t nq) {
    return static_cast<unsigned>(kXcds * nq * ((njb + kXcds - 1) / kXcds));
  };
  double* part = static_cast<double*>(work);
  // The triangle form, in the number nq of splits that takes it least time, where
  // that is less than the full form's: rounds of kSlots resident blocks (a last one of
  // a block per CU at most is shorter) times the conditions a block's K loops pass,
  // n in the full form, those of the longest split's row blocks in this one, and
  // kSymCost for the triangle's own launch.  The workspace, 2 nib N doubles, has to
  // hold the triangle and w beside the partial sums (from about n^2 / (2 nib) targets,
  // 6.5e4 at n = 1000).  Not for one row block, whose K loops are the full form's.
  // Full and triangle form: n = 300, N = 1e5 0.49 and 0.78 ms in two unequal splits;
  // n = 385, N = 2.5e5 1.86 and 1.45.
  const int64_t ld = (n + kKK - 1) / kKK * kKK;
  const int64_t tri = ld * ld + kKI + n;  // kKI: the last row's loads reach past it
  auto rounds = [](int64_t b) {
    const int64_t r = b % kSlots;
    return static_cast<double>(b / kSlots) + (r == 0 ? 0.0 : (2 * r <= kSlots ? 0.6 : 1.0));
  };
  int64_t nq = 0;
  double least = kTriSure * rounds(njb * nib) * static_cast<double>(n);
  for (int64_t t = 1; nib > 1 && t <= std::min<int64_t>(nib, (kTriBlocks + njb - 1) / njb); ++t) {
    if (tri > 2 * N * (t > 1 ? nib - t : nib)) continue;
    int64_t longest = 0;
    for (int64_t q = 0; q < t; ++q) {
      int64_t k = 0;
      for (int64_t turn = 0; turn * t < nib; ++turn) {
        const int64_t ib = turn * t + (turn & 1 ? t - 1 - q : q);
        if (ib < nib) k += std::min((ib + 1) * kKI, n);
      }
      longest = std::max(longest, k);
    }
    const double cost = rounds(njb * t) * static_cast<double>(longest) + kSymCost;
    if (cost < least) {
      least = cost;
      nq = t;
    }
  }
  if (nq > 0) {
    double* st = part + (nq > 1 ? 2 * nq * N : 0);
    double* w = st + ld * ld + kKI;
    const int64_t nt = (ld + kSymTile - 1) / kSymTile;
    const int seg = static_cast<int>(std::max<int64_t>(n / 3 / 64 * 64, 64));
    k_krige_sym<<<static_cast<unsigned>(nt * nt + wb), 256, 0, s>>>(n, ld, nt, mat, cond, st, w);
    k_krige_tiles<TRIANGLE><<<blocks(nq), 256, 0, s>>>(n, N, st, ld, vecs, vld, w, nib,
                                                   static_cast<int>(nq), static_cast<int>(njb),
                                                   seg, part, field, error);
    if (nq > 1) k_krige_sum<true><<<jb, 256, 0, s>>>(N, static_cast<int>(nq), part, field, error);
    k_krige_tiles<REDO><<<blocks(1), 256, 0, s>>>(n, N, mat, n, vecs, vld, cond, nib, 1,
                                                  static_cast<int>(njb), static_cast<int>(n),
                                                  nullptr, field, error);
    return hipGetLastError();
  }
  if (nib > 0) {
    auto* full = n > kKI / 2 ? k_krige_tiles<FULL> : k_krige_tiles<FULL, true>;
    full<<<blocks(nib), 256, 0, s>>>(n, N, mat, n, vecs, vld, cond, nib, nib,
                                     static_cast<int>(njb), static_cast<int>(n), part, field,
                                     error);
  }
  k_krige_sum<false><<<jb, 256, 0, s>>>(N, nib, part, field, error);
  return hipGetLastError();
}

}  // namespace gsc
