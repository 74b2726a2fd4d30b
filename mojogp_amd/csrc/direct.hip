// Kernel-matrix products from per-dimension differences of the scaled
// coordinates (no Gram form): Matern-1/2, point sets whose norms exceed the
// Gram bound, and input dimensions beyond the tile path.
//
// Reference behaviour (caspbian/mojogp):
//   fused_forward_matvec_ncols  mojogp/codegen_engine/emit/gpu_kernel.py:151-260
//   fused_cross_matvec_ncols    mojogp/codegen_engine/emit/gpu_kernel.py:487-565
//
// Per pair 2 d + ~5 VALU instructions form the fp32 value, which enters the
// product with the right-hand sides in fp64: as an operand of
// v_mfma_f64_16x16x4_f64 or, for up to 4 right-hand sides, of VALU FMAs.
// Issue bound: at d = 5 the value costs ~62 cycles per 64 pairs, the matrix
// instruction 64, so 200 us (side by side) to 320 us for n = 20011 one-sided;
// measured 411 us with the reduction (11 right-hand sides, Matern-1/2) and 373
// us over unordered pairs, against 18.7 ms for one row per thread (79
// workgroups, run-time dimension loops).
//
// fp32 matrix sums (64 columns before fp64) took 330 and 263 us, but lost
// accuracy that one fp64 addition per product had: relative error of rough
// right-hand sides, one addition / fp32 sums / here: d = 1, n = 3001, 11
// columns 7.7e-8 / 1.8e-7 / 5.8e-8; d = 5, n = 12807 1.4e-7 / 2.2e-7 / 1.4e-7;
// of a predictive mean (alpha's terms cancel), n = 3001 3.6e-6 / 6.9e-6 /
// 3.0e-6.
#include "kval.h"
#include "matvec.h"
#include "sym_common.h"

#include <algorithm>
#include <vector>

namespace mgp {

namespace {

typedef float f4 __attribute__((ext_vector_type(4)));
typedef double d4 __attribute__((ext_vector_type(4)));

constexpr int kDiffTile = 64;    // column points per LDS tile
constexpr int kDiffWaves = 4;    // waves per workgroup

// Right-hand sides a kernel form carries: VALU forms 1 and 4, matrix-core
// forms 16 and 64.
enum DiffForm { kDiff1 = 0, kDiff4, kDiff16, kDiff64, kDiffForms };
constexpr int kDiffCols[kDiffForms] = {1, 4, 16, 64};

// 16-row tiles per wave: row coordinates (R x D) and accumulators stay in
// registers with at least 3 waves per SIMD (n = 30000, 16 right-hand sides,
// symmetric: d = 16 1.05 ms with 4, 0.98 ms with 2; d = 5 0.74 and 0.76 ms; one
// right-hand side at d = 24 1.21 and 1.12 ms).
constexpr int diff_rows(int D, int form) {
  return D > 10 || form == kDiff64 ? 2 : 4;
}

// os tot + noise v in fp64, rounded once (v = 0 where no noise is added).
__device__ __forceinline__ float diff_epilogue(double tot, float os, float noise, float v) {
  return (float)((double)os * tot + (double)noise * (double)v);
}

// Sums over the columns [y tps 64, (y + 1) tps 64) of split y, for rows
// i0 + 16 r + lane%16 of each wave.  Step s of a column tile: lane l evaluates
// the pairs (row 16 r + l%16, column 4 s + l/16), r < R, from one LDS read of
// the column point; they are the A operand of v_mfma_f64_16x16x4_f64 with
// B = V[column][l%16], whose result holds rows 16 r + 4 q + l/16 of right-hand
// side l%16.  Products and sums in fp64 throughout.
// part != nullptr: part[(y nc + c) m + i] = the fp64 sums; else (one split)
// the epilogue out = os sum (+ noise V).
template <int KIND, int D, int FORM>
__global__ __launch_bounds__(64 * kDiffWaves) void k_diff_tile(
    const float* __restrict__ Zr, int64_t m, const float* __restrict__ Zc, int64_t n, int d,
    const float* __restrict__ V, int nc, int64_t tps, float os, float noise, int add_noise,
    float lim, double* __restrict__ part, float* __restrict__ out) {
  constexpr int R = diff_rows(D, FORM);
  constexpr bool MFMA = FORM >= kDiff16;
  constexpr int NC = kDiffCols[FORM];
  constexpr int G = MFMA ? NC / 16 : 1;          // 16-column groups
  constexpr int DS = D <= 2 ? D : (D + 3) / 4 * 4;  // LDS stride of a column point
  __shared__ __align__(16) float sx[kDiffTile * DS];
  __shared__ __align__(16) float sv[kDiffTile * NC];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lm = lane & 15, lq = lane >> 4;
  const int64_t i0 = ((int64_t)blockIdx.x * kDiffWaves + wave) * (16 * R);

  float xi[R][D];
#pragma unroll
  for (int r = 0; r < R; ++r) {
    const int64_t i = i0 + 16 * r + lm;
#pragma unroll
    for (int k = 0; k < D; ++k) xi[r][k] = (i < m && k < d) ? Zr[i * d + k] : 0.0f;
  }
  d4 am[R][G];        // matrix forms
  double acc[R][NC];  // VALU forms: this lane's columns
#pragma unroll
  for (int r = 0; r < R; ++r) {
#pragma unroll
    for (int g = 0; g < G; ++g) am[r][g] = d4{0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int c = 0; c < NC; ++c) acc[r][c] = 0.0;
  }

  const int64_t tiles = (n + kDiffTile - 1) / kDiffTile;
  const int64_t t0 = (int64_t)blockIdx.y * tps, t1 = min(tiles, t0 + tps);
  for (int64_t t = t0; t < t1; ++t) {
    const int64_t j0 = t * kDiffTile;
    const int cnt = (int)min((int64_t)kDiffTile, n - j0);
    __syncthreads();
    // columns past n: zero coordinates and zero right-hand sides
    for (int q = threadIdx.x; q < kDiffTile * D; q += 64 * kDiffWaves) {
      const int jj = q / D, k = q - jj * D;
      sx[jj * DS + k] = (jj < cnt && k < d) ? Zc[(j0 + jj) * d + k] : 0.0f;
    }
    for (int q = threadIdx.x; q < kDiffTile * NC; q += 64 * kDiffWaves) {
      const int c = q / kDiffTile, jj = q - c * kDiffTile;
      sv[jj * NC + c] = (jj < cnt && c < nc) ? V[(int64_t)c * n + j0 + jj] : 0.0f;
    }
    __syncthreads();
    const int steps = (cnt + 3) / 4;
#pragma unroll 2
    for (int s = 0; s < steps; ++s) {
      const int jj = 4 * s + lq;
      float xj[DS];
      if constexpr (D <= 2) {
#pragma unroll
        for (int k = 0; k < D; ++k) xj[k] = sx[jj * DS + k];
      } else {
#pragma unroll
        for (int k = 0; k < DS; k += 4) {
          const f4 x = *reinterpret_cast<const f4*>(&sx[jj * DS + k]);
#pragma unroll
          for (int e = 0; e < 4; ++e) xj[k + e] = x[e];
        }
      }
      double v[MFMA ? G : NC];
      if constexpr (MFMA) {
#pragma unroll
        for (int g = 0; g < G; ++g) v[g] = (double)sv[jj * NC + 16 * g + lm];
      } else {
#pragma unroll
        for (int c = 0; c < NC; ++c) v[c] = (double)sv[jj * NC + c];
      }
#pragma unroll
      for (int r = 0; r < R; ++r) {
        float r2 = 0.0f;
#pragma unroll
        for (int k = 0; k < D; ++k) {
          const float df = xi[r][k] - xj[k];
          r2 = fmaf(df, df, r2);
        }
        const double kv = (double)kval<KIND>(r2, lim);
        if constexpr (MFMA) {
#pragma unroll
          for (int g = 0; g < G; ++g)
            if (g == 0 || 16 * g < nc)  // (uniform) groups past nc hold no right-hand side
              am[r][g] = __builtin_amdgcn_mfma_f64_16x16x4f64(kv, v[g], am[r][g], 0, 0, 0);
        } else {
#pragma unroll
          for (int c = 0; c < NC; ++c) acc[r][c] = fma(kv, v[c], acc[r][c]);
        }
      }
    }
  }

  auto put = [&](int c, int64_t i, double tot) __attribute__((always_inline)) {
    if (c >= nc || i >= m) return;
    if (part) {
      part[((int64_t)blockIdx.y * nc + c) * m + i] = tot;
    } else {
      out[(int64_t)c * m + i] =
          diff_epilogue(tot, os, noise, add_noise ? V[(int64_t)c * m + i] : 0.0f);
    }
  };
#pragma unroll
  for (int r = 0; r < R; ++r) {
    if constexpr (MFMA) {
#pragma unroll
      for (int g = 0; g < G; ++g)
#pragma unroll
        for (int q = 0; q < 4; ++q) put(16 * g + lm, i0 + 16 * r + 4 * q + lq, am[r][g][q]);
    } else {
      // the four lane groups hold the row's columns 4 s + l/16: fold them
#pragma unroll
      for (int c = 0; c < NC; ++c) {
        double tot = acc[r][c];
        tot += __shfl_xor(tot, 16);
        tot += __shfl_xor(tot, 32);
        if (lq == 0) put(c, i0 + 16 * r + lm, tot);
      }
    }
  }
}

// out[c][i] = os sum_y part[y][c][i] (+ noise V[c][i]), splits in order.
__global__ void k_diff_reduce(const double* __restrict__ part, int splits, int64_t total,
                              float os, float noise, int add_noise, const float* __restrict__ V,
                              float* __restrict__ out) {
  const int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (idx >= total) return;
  double tot = 0.0;
#pragma unroll 4
  for (int s = 0; s < splits; ++s) tot += part[(int64_t)s * total + idx];
  out[idx] = diff_epilogue(tot, os, noise, add_noise ? V[idx] : 0.0f);
}

using DiffFn = void (*)(const float*, int64_t, const float*, int64_t, int, const float*, int,
                        int64_t, float, float, int, float, double*, float*);

struct DiffKernel {
  DiffFn fn;
  int rows;  // rows per workgroup
};

// Every dimension up to 6, then the steps at which a padded dimension costs
// at most a quarter of the value's instructions.
template <int KIND, int FORM>
DiffKernel pick_diff_d(int d) {
#define MGP_DIFF_CASE(DV) \
  if (d <= DV) return {k_diff_tile<KIND, DV, FORM>, 16 * diff_rows(DV, FORM) * kDiffWaves};
  MGP_DIFF_CASE(1)
  MGP_DIFF_CASE(2)
  MGP_DIFF_CASE(3)
  MGP_DIFF_CASE(4)
  MGP_DIFF_CASE(5)
  MGP_DIFF_CASE(6)
  MGP_DIFF_CASE(8)
  MGP_DIFF_CASE(10)
  MGP_DIFF_CASE(12)
  MGP_DIFF_CASE(16)
  MGP_DIFF_CASE(20)
  MGP_DIFF_CASE(24)
  MGP_DIFF_CASE(32)
#undef MGP_DIFF_CASE
  return {nullptr, 0};
}

template <int KIND>
DiffKernel pick_diff_form(int form, int d) {
  switch (form) {
    case kDiff1: return pick_diff_d<KIND, kDiff1>(d);
    case kDiff4: return pick_diff_d<KIND, kDiff4>(d);
    case kDiff16: return pick_diff_d<KIND, kDiff16>(d);
    default: return pick_diff_d<KIND, kDiff64>(d);
  }
}

DiffKernel pick_diff(int kind, int form, int d) {
  switch (kind) {
    case KIND_RBF: return pick_diff_form<KIND_RBF>(form, d);
    case KIND_MATERN12: return pick_diff_form<KIND_MATERN12>(form, d);
    case KIND_MATERN32: return pick_diff_form<KIND_MATERN32>(form, d);
    default: return pick_diff_form<KIND_MATERN52>(form, d);
  }
}

// Column splits of a launch of row_blocks workgroups: the chip holds `slots`
// workgroups at once, so a launch takes ceil(blocks / slots) rounds of
// (tiles per split + about half a tile of set-up); every split's fp64 partials
// are written once and read once (about 1/40 of a tile's time per split and
// slot-filling of rows, which only keeps tiny splits apart).
int64_t diff_splits(int64_t row_blocks, int64_t tiles, int64_t slots) {
  int64_t best = 1;
  double best_cost = 0.0;
  for (int64_t s = 1; s <= std::min<int64_t>(tiles, 64); ++s) {
    const int64_t tps = ceil_div(tiles, s);
    if (s > 1 && ceil_div(tiles, s - 1) == tps) continue;
    const int64_t real = ceil_div(tiles, tps);
    const double rounds = (double)ceil_div(row_blocks * real, slots);
    const double cost =
        rounds * ((double)tps + 0.5) + 0.025 * (double)real * (double)row_blocks / 64.0;
    if (s == 1 || cost < best_cost) {
      best_cost = cost;
      best = real;
    }
  }
  return best;
}

// ---------------------------------------------------------------------------
// Square products with 5 to 16 right-hand sides: every unordered pair is formed
// once.  Blocks of 64 R points (4 waves of R row tiles); row block b takes
// stages (64 columns each) of its own block and of the column blocks (b +
// delta) mod nb of the cyclic half (sym_span).  Per 16 x 16 tile a lane
// evaluates the pairs (row lane%16, columns 4 (lane/16) + s), the A operands of
// out_I += K V_J; their rows go through a wave-private LDS tile (stride 20:
// conflict-free both ways) and come back as the A operands of out_J += K^T V_I
// with the rows' right-hand sides in registers, both in fp64 (as k_diff_tile).
// The waves' transposed sums are added in LDS and written per stage.  The
// value's 2 d + 7 instructions are paid once for two entries, the matrix
// instructions (64 cycles per 4 columns of a tile) per entry.  Matern-1/2, 16
// right-hand sides, one-sided -> here: d = 1 n = 30000 685 -> 649 us; d = 5 n =
// 20011 417 -> 378, n = 30000 871 -> 737; d = 16 n = 30000 1177 -> 982.
// fwd[(split 16 + c) npad + i] (one rounding per split, as tp's per stage),
// tp[((b hmax + delta - 1) BLK + j) 16 + c].
// ---------------------------------------------------------------------------
constexpr int kDiffSymStage = 64;
constexpr int diff_sym_rows(int D) { return D > 10 ? 2 : 4; }

template <int KIND, int D>
__global__ __launch_bounds__(64 * kDiffWaves) void k_diff_sym(
    const float* __restrict__ Z, int64_t n, int d, const float* __restrict__ V, int nc,
    int64_t nb, int64_t sps, int64_t hmax, float lim, float* __restrict__ fwd,
    float* __restrict__ tp) {
  constexpr int R = diff_sym_rows(D), BLK = 64 * R, ST = kDiffSymStage, VS = 20;
  constexpr int DS = D <= 2 ? D : (D + 3) / 4 * 4;
  constexpr int per = BLK / ST;
  __shared__ __align__(16) float sx[ST * DS];
  __shared__ __align__(16) float sv[ST * VS];
  __shared__ __align__(16) float tsc[kDiffWaves][2][16 * VS];
  __shared__ d4 tbuf[kDiffWaves][ST / 16][64];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lm = lane & 15, lq = lane >> 4;
  const int64_t b = blockIdx.x, split = blockIdx.y, npad = nb * BLK;
  const int64_t i0 = b * BLK + wave * (16 * R);
  float xi[R][D];
  double vr[R][4];
#pragma unroll
  for (int r = 0; r < R; ++r) {
    const int64_t i = i0 + 16 * r + lm;
#pragma unroll
    for (int k = 0; k < D; ++k) xi[r][k] = (i < n && k < d) ? Z[i * d + k] : 0.0f;
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      const int64_t ii = i0 + 16 * r + 4 * lq + s;
      vr[r][s] = (ii < n && lm < nc) ? (double)V[(int64_t)lm * n + ii] : 0.0;
    }
  }
  d4 acc[R];
#pragma unroll
  for (int r = 0; r < R; ++r) acc[r] = d4{0.0, 0.0, 0.0, 0.0};
  const int64_t g0 = split * sps, g1 = min(g0 + sps, (sym_span(b, nb) + 1) * per);
  for (int64_t g = g0; g < g1; ++g) {
    const int64_t dl = g / per;
    int64_t J = b + dl;
    if (J >= nb) J -= nb;
    const int64_t j0 = J * BLK + (g % per) * ST;
    // (the previous stage's operands are free: its second barrier)
    for (int q = threadIdx.x; q < ST * D; q += 64 * kDiffWaves) {
      const int jj = q / D, k = q - jj * D;
      sx[jj * DS + k] = (j0 + jj < n && k < d) ? Z[(j0 + jj) * d + k] : 0.0f;
    }
    for (int q = threadIdx.x; q < ST * 16; q += 64 * kDiffWaves) {
      const int c = q / ST, jj = q - c * ST;
      sv[jj * VS + c] = (c < nc && j0 + jj < n) ? V[(int64_t)c * n + j0 + jj] : 0.0f;
    }
    __syncthreads();
#pragma unroll 1
    for (int ct = 0; ct < ST / 16; ++ct) {
      d4 d2 = d4{0.0, 0.0, 0.0, 0.0};
      float kv[R][4];
#pragma unroll
      for (int s = 0; s < 4; ++s) {
        const int jj = 16 * ct + 4 * lq + s;
        float xj[DS];
        if constexpr (D <= 2) {
#pragma unroll
          for (int k = 0; k < D; ++k) xj[k] = sx[jj * DS + k];
        } else {
#pragma unroll
          for (int k = 0; k < DS; k += 4) {
            const f4 x = *reinterpret_cast<const f4*>(&sx[jj * DS + k]);
#pragma unroll
            for (int e = 0; e < 4; ++e) xj[k + e] = x[e];
          }
        }
        const double v = (double)sv[jj * VS + lm];
#pragma unroll
        for (int r = 0; r < R; ++r) {
          float r2 = 0.0f;
#pragma unroll
          for (int k = 0; k < D; ++k) {
            const float df = xi[r][k] - xj[k];
            r2 = fmaf(df, df, r2);
          }
          kv[r][s] = kval<KIND>(r2, lim);
          acc[r] = __builtin_amdgcn_mfma_f64_16x16x4f64((double)kv[r][s], v, acc[r], 0, 0, 0);
        }
      }
      if (dl > 0) {
#pragma unroll
        for (int r = 0; r < R; ++r) {
          float* sc = tsc[wave][r & 1];
          *reinterpret_cast<f4*>(sc + lm * VS + 4 * lq) =
              f4{kv[r][0], kv[r][1], kv[r][2], kv[r][3]};
          wave_lds_sync();  // (the other buffer's reads, too, stay before its next store)
#pragma unroll
          for (int s = 0; s < 4; ++s)
            d2 = __builtin_amdgcn_mfma_f64_16x16x4f64((double)sc[(4 * lq + s) * VS + lm], vr[r][s],
                                                      d2, 0, 0, 0);
        }
        tbuf[wave][ct][lane] = d2;
      }
    }
    __syncthreads();
    if (dl > 0) {
      // lane of column tile ct: columns 4 q + lane/16, right-hand side lane%16
      float* dst = tp + ((b * hmax + dl - 1) * BLK + (g % per) * ST) * 16;
      for (int q = threadIdx.x; q < ST * 4; q += 64 * kDiffWaves) {
        const int ct = q >> 6, ln = q & 63;
        double t[4] = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
        for (int w = 0; w < kDiffWaves; ++w)
#pragma unroll
          for (int k = 0; k < 4; ++k) t[k] += tbuf[w][ct][ln][k];
#pragma unroll
        for (int k = 0; k < 4; ++k)
          dst[(16 * ct + 4 * k + (ln >> 4)) * 16 + (ln & 15)] = (float)t[k];
      }
    }
  }
#pragma unroll
  for (int r = 0; r < R; ++r)
#pragma unroll
    for (int q = 0; q < 4; ++q)
      fwd[(split * 16 + lm) * npad + i0 + 16 * r + 4 * q + lq] = (float)acc[r][q];
}

// out[c][j] = os (split sums + the transposed partials of the row blocks that
// formed j's column block, in delta order) + noise V: fp64, rounded once.
// Four threads per point own four right-hand sides each; unformed slots (nb
// even, the last delta) are read and dropped by a select.
__global__ __launch_bounds__(256) void k_diff_sym_reduce(
    const float* __restrict__ fwd, int splits, const float* __restrict__ tp, int block,
    int64_t nb, int64_t hmax, int64_t n, int nc, float os, float noise,
    const float* __restrict__ V, float* __restrict__ out) {
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int64_t j = t >> 2;
  const int c4 = 4 * (int)(t & 3);
  if (j >= n) return;
  const int64_t npad = nb * block;
  double tot[4] = {0.0, 0.0, 0.0, 0.0};
  for (int y = 0; y < splits; ++y)
#pragma unroll
    for (int e = 0; e < 4; ++e) tot[e] += fwd[((int64_t)y * 16 + c4 + e) * npad + j];
  const int64_t J = j / block, jl = j - J * block;
  auto slot = [&](int64_t dl, bool& formed) __attribute__((always_inline)) {
    int64_t bb = J - dl;
    bb += bb < 0 ? nb : 0;
    formed = dl <= sym_span(bb, nb);
    return __builtin_nontemporal_load(reinterpret_cast<const f4*>(
        tp + ((bb * hmax + dl - 1) * block + jl) * 16 + c4));
  };
  int64_t dl = 1;
  for (; dl + 8 <= hmax + 1; dl += 8) {
    f4 v[8];
    bool ok[8];
#pragma unroll
    for (int q = 0; q < 8; ++q) v[q] = slot(dl + q, ok[q]);
#pragma unroll
    for (int q = 0; q < 8; ++q)
#pragma unroll
      for (int e = 0; e < 4; ++e) tot[e] += ok[q] ? (double)v[q][e] : 0.0;
  }
  for (; dl <= hmax; ++dl) {
    bool ok;
    const f4 v = slot(dl, ok);
#pragma unroll
    for (int e = 0; e < 4; ++e) tot[e] += ok ? (double)v[e] : 0.0;
  }
#pragma unroll
  for (int e = 0; e < 4; ++e)
    if (c4 + e < nc) {
      const int64_t idx = (int64_t)(c4 + e) * n + j;
      out[idx] = diff_epilogue(tot[e], os, noise, V[idx]);
    }
}

using DiffSymFn = void (*)(const float*, int64_t, int, const float*, int, int64_t, int64_t,
                           int64_t, float, float*, float*);
struct DiffSymKernel {
  DiffSymFn fn;
  int block;
};

template <int KIND>
DiffSymKernel pick_diff_sym_d(int d) {
#define MGP_DIFF_CASE(DV) \
  if (d <= DV) return {k_diff_sym<KIND, DV>, 64 * diff_sym_rows(DV)};
  MGP_DIFF_CASE(1)
  MGP_DIFF_CASE(2)
  MGP_DIFF_CASE(3)
  MGP_DIFF_CASE(4)
  MGP_DIFF_CASE(5)
  MGP_DIFF_CASE(6)
  MGP_DIFF_CASE(8)
  MGP_DIFF_CASE(10)
  MGP_DIFF_CASE(12)
  MGP_DIFF_CASE(16)
  MGP_DIFF_CASE(20)
  MGP_DIFF_CASE(24)
  MGP_DIFF_CASE(32)
#undef MGP_DIFF_CASE
  return {nullptr, 0};
}

DiffSymKernel pick_diff_sym(int kind, int d) {
  switch (kind) {
    case KIND_RBF: return pick_diff_sym_d<KIND_RBF>(d);
    case KIND_MATERN12: return pick_diff_sym_d<KIND_MATERN12>(d);
    case KIND_MATERN32: return pick_diff_sym_d<KIND_MATERN32>(d);
    default: return pick_diff_sym_d<KIND_MATERN52>(d);
  }
}

// Half the values pay for the transposed products, their partial sums and the
// reduction from here on, earlier where a value costs more (one-sided ->
// symmetric us, Matern-1/2, 11 right-hand sides: d = 1 n = 14000 171 -> 183,
// 16000 217 -> 215, 30000 679 -> 643; d = 3 11000 133 -> 141, 14000 198 -> 194;
// d = 5 11000 144 -> 150, 12000 169 -> 152; d = 10 7000 90 -> 102, 8000 108 ->
// 106, 9000 144 -> 127; d = 16 5000 84 -> 81, 6000 95 -> 84, 7000 110 -> 107; d =
// 24 5000 90 -> 96, 6000 116 -> 100).  Up to 4 right-hand sides the one-sided
// kernel spends no matrix instructions (n = 30000, d = 16, 4 columns: 865 ->
// 942).
constexpr int64_t kDiffSymMin = 5500;
constexpr int64_t kDiffSymBase = 15500, kDiffSymPerDim = 750;
// 17 to 32 right-hand sides: two groups of the 64-column form evaluate as many
// pairs as two symmetric passes and sum fewer partials, but keep fewer waves on
// a CU.  Two groups -> two passes, 32 columns, us: d = 1 n = 14000 370 -> 376,
// 20011 709 -> 652, 40000 2686 -> 2154; d = 5 12000 315 -> 294, 20011 799 ->
// 743, 40000 2899 -> 2429; d = 16 9000 256 -> 281, 20011 1016 -> 955, 40000 3711
// -> 3546; d = 24 20011 1172 -> 1270.
constexpr int kDiffPairMaxDim = 16;
constexpr int64_t kDiffPairMin = 20000;
constexpr double kDiffSymMaxBytes = 8e9;  // of transposed partials (at most n^2 / 4)

bool diff_sym_route(const MatvecArgs& a, const PackedPoints& rows, const PackedPoints& cols,
                    int d, int nc, const MatvecWorkspace& ws) {
  if (!a.square || &rows != &cols || a.m != a.n || ws.arena != nullptr || nc > 16) return false;
  if ((double)a.n * (double)a.n / 4 > kDiffSymMaxBytes) return false;
  const int mode = sym_switch();
  if (mode >= 0) return mode == 1;
  return nc >= 5 && a.n >= kDiffSymMin && a.n + kDiffSymPerDim * d >= kDiffSymBase;
}

// False, with nothing launched, where its partial sums do not fit the device.
bool diff_sym_matvec(const MatvecArgs& a, const PackedPoints& pts, int d, const float* V, int nc,
                     float* out, MatvecWorkspace& ws, int cus, hipStream_t st) {
  const DiffSymKernel k = pick_diff_sym(a.kind, d);
  MGP_REQUIRE(k.fn != nullptr, "no difference kernel for this shape");
  int per_cu = 0;
  MGP_HIP_CHECK(hipOccupancyMaxActiveBlocksPerMultiprocessor(
      &per_cu, reinterpret_cast<const void*>(k.fn), 64 * kDiffWaves, 0));
  const int64_t n = a.n, nb = ceil_div(n, (int64_t)k.block), hmax = nb / 2;
  const int64_t stages = (hmax + 1) * (k.block / kDiffSymStage);
  const int64_t slots = (int64_t)std::max(cus, 1) * std::max(per_cu, 1);
  // rounds of (stages a workgroup + about half of one of set-up)
  int64_t splits = 1;
  double best = 0.0;
  for (int64_t s = 1; s <= std::min<int64_t>(stages, 64); ++s) {
    const int64_t sps = ceil_div(stages, s);
    if (ceil_div(stages, sps) != s) continue;
    const double cost = (double)ceil_div(nb * s, slots) * ((double)sps + 0.5) + 0.05 * (double)s;
    if (s == 1 || cost < best) {
      best = cost;
      splits = s;
    }
  }
  float* fwd = ws.partial.try_ensure((size_t)splits * 16 * nb * k.block);
  float* tp = ws.sym_tp.try_ensure((size_t)std::max<int64_t>(nb * hmax, 1) * k.block * 16);
  if (fwd == nullptr || tp == nullptr) return false;
  hipLaunchKernelGGL(k.fn, dim3((unsigned)nb, (unsigned)splits), dim3(64 * kDiffWaves), 0, st,
                     pts.z.ptr, n, d, V, nc, nb, ceil_div(stages, splits), hmax, pts.exp2_limit,
                     fwd, tp);
  hipLaunchKernelGGL(k_diff_sym_reduce, dim3((unsigned)ceil_div(4 * n, 256)), dim3(256), 0, st, fwd,
                     (int)splits, tp, k.block, nb, hmax, n, nc, a.outputscale, a.noise, V, out);
  MGP_HIP_CHECK(hipGetLastError());
  return true;
}

}  // namespace

void direct_matvec(const MatvecArgs& a, const PackedPoints& rows, const PackedPoints& cols, int d,
                   const float* V_dev, float* out_dev, MatvecWorkspace& ws, hipStream_t st) {
  MGP_REQUIRE(d >= 1 && d <= 32, "direct path supports input dimension <= 32");
  if (a.m <= 0 || a.ncols <= 0) return;
  int dev = 0, cus = 0;
  MGP_HIP_CHECK(hipGetDevice(&dev));
  MGP_HIP_CHECK(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev));
  const int64_t tiles = ceil_div(std::max<int64_t>(a.n, 1), kDiffTile);
  for (int c0 = 0; c0 < a.ncols;) {
    // up to 4 columns on the VALU (a value then costs at most 4 FMAs against
    // the 32 cycles of its matrix instruction), up to 16 in one matrix
    // group; up to four groups share the values of a wider product
    const int left = a.ncols - c0;
    int form = left == 1 ? kDiff1 : left <= 4 ? kDiff4 : left <= 16 ? kDiff16 : kDiff64;
    if (left > 16 && left <= 32 && d <= kDiffPairMaxDim && a.n >= kDiffPairMin &&
        diff_sym_route(a, rows, cols, d, 16, ws))
      form = kDiff16;
    const int nc = std::min(kDiffCols[form], left);
    if (diff_sym_route(a, rows, cols, d, nc, ws) &&
        diff_sym_matvec(a, rows, d, V_dev + (int64_t)c0 * a.n, nc, out_dev + (int64_t)c0 * a.m, ws,
                        cus, st)) {
      c0 += nc;
      continue;
    }
    const DiffKernel k = pick_diff(a.kind, form, d);
    MGP_REQUIRE(k.fn != nullptr, "no difference kernel for this shape");
    const int64_t row_blocks = ceil_div(a.m, k.rows);
    int per_cu = 0;
    MGP_HIP_CHECK(hipOccupancyMaxActiveBlocksPerMultiprocessor(
        &per_cu, reinterpret_cast<const void*>(k.fn), 64 * kDiffWaves, 0));
    int64_t splits =
        diff_splits(row_blocks, tiles, (int64_t)std::max(cus, 1) * std::max(per_cu, 1));
    const int64_t total = (int64_t)nc * a.m;
    double* part = nullptr;
    if (ws.arena != nullptr) {
      // fixed arena: as many splits as its bytes hold, unsplit without partials
      splits = std::min<int64_t>(splits, (int64_t)(ws.arena_bytes / (sizeof(double) * total)));
      if (splits > 1) part = reinterpret_cast<double*>(ws.arena);
    } else if (splits > 1) {
      part = ws.direct_part.ensure((size_t)splits * total);
    }
    const int64_t tps = ceil_div(tiles, std::max<int64_t>(splits, 1));
    splits = ceil_div(tiles, tps);
    const float* Vc = V_dev + (int64_t)c0 * a.n;
    float* outc = out_dev + (int64_t)c0 * a.m;
    const int add = a.square ? 1 : 0;
    hipLaunchKernelGGL(k.fn, dim3((unsigned)row_blocks, (unsigned)splits), dim3(64 * kDiffWaves),
                       0, st, rows.z.ptr, a.m, cols.z.ptr, a.n, d, Vc, nc, tps, a.outputscale,
                       a.noise, add, cols.exp2_limit, part, outc);
    MGP_HIP_CHECK(hipGetLastError());
    if (part) {
      hipLaunchKernelGGL(k_diff_reduce, dim3((unsigned)ceil_div(total, 256)), dim3(256), 0, st,
                         part, (int)splits, total, a.outputscale, a.noise, add, Vc, outc);
      MGP_HIP_CHECK(hipGetLastError());
    }
    c0 += nc;
  }
}

}  // namespace mgp
