// Gradient traces of single radial kernels from per-dimension differences:
// Matern-1/2, point sets beyond the Gram bound, more than 16 dimensions, and
// models below the matrix-core trace's size (matvec.hip k_grad_sym).
//
// Reference behaviour (caspbian/mojogp): the gradient products
// fused_all_gradients_matvec (codegen_engine/emit/gpu_kernel.py:382-484)
// contracted with the BBMM weight columns.
#include "kval.h"
#include "matvec.h"
#include "sym_common.h"

#include <algorithm>
#include <vector>

namespace mgp {

namespace {

typedef float f4 __attribute__((ext_vector_type(4)));

constexpr int kGpBlock = 128;            // points per block (rows and columns)
constexpr int kGpR = 2;                  // 16-row tiles per wave, 4 waves
constexpr int kGpCols = 16;              // factor columns per pass
constexpr int kGpStride = kGpBlock + 16; // LDS stride of a factor column
constexpr int kGpFlush = 2;              // 16-column tiles between fp64 flushes

// k / os and the lengthscale factor h (dk/dl_q = os h dz_q^2 / (s^2 l_q)) from
// the scaled squared distance.
template <int KIND, bool ARD>
__device__ __forceinline__ void value_and_h(float r2, float& kv, float& h) {
  if constexpr (KIND == KIND_RBF) {
    kv = __builtin_amdgcn_exp2f(-r2);  // not clamped
    h = kv;
  } else if constexpr (KIND == KIND_MATERN12) {
    // h = log2(e) k / r with the reference's floored r = sqrt(r^2 + 1e-20);
    // the exponent is clamped for ARD only (exp2_limit)
    const float u = __builtin_amdgcn_sqrtf(r2);
    kv = __builtin_amdgcn_exp2f(ARD ? -fminf(u, kExp2Clamp) : -u);
    h = kLog2e * kv / __builtin_amdgcn_sqrtf(r2 + kM12RFloor);
  } else if constexpr (KIND == KIND_MATERN32) {
    const float u = __builtin_amdgcn_sqrtf(r2);
    const float e = __builtin_amdgcn_exp2f(-fminf(u, kExp2Clamp));
    kv = fmaf(u, kLn2, 1.0f) * e;
    h = 3.0f * e;
  } else {
    const float u = __builtin_amdgcn_sqrtf(r2);
    const float e = __builtin_amdgcn_exp2f(-fminf(u, kExp2Clamp));
    kv = fmaf(u, fmaf(u, kM52B, kM52A), 1.0f) * e;
    h = (5.0f / 3.0f) * fmaf(u, kLn2, 1.0f) * e;
  }
}

// part[(y gx + x) nterms + q] = the workgroup's share of
//   sum_ab W_ab h_ab dz_abq^2 (ARD: q < d; isotropic: the sum over q), then
//   sum_ab W_ab k_ab / os,                W_ab = sum_c Lf[c][a] Rf[c][b].
// h, dz^2 and k are symmetric, so each unordered pair is formed once with
// W_ab + W_ba: blocks of 128 points, row block b taking the column blocks
// (b + delta) mod nb of the cyclic half (sym_span), its own with weight 1/2.
// W_ab + W_ba of a 16 x 16 tile comes from the fp32 matrix cores (four factor
// columns an instruction); its result q belongs to the pair (column 4
// (lane/16) + q, row lane%16), so a lane keeps its rows in registers and
// reads columns from LDS.  VALU bound: 4 d + ~10 instructions an unordered
// pair; the pair loop it replaces spent 3 d + 28 on each ordered one, on one
// row per thread and at least 1024 columns a workgroup (n = 1001, d = 5: 579
// -> 60 us a trace with the host copies; n = 10007: 611 -> 160; n = 25000, d =
// 16: 1.67 -> 1.16 ms).
template <int KIND, int D, bool ARD>
__global__ __launch_bounds__(256) void k_grad_pair(
    const float* __restrict__ Z, int64_t n, int d, const float* __restrict__ Lf,
    const float* __restrict__ Rf, int ncols, int c0, int64_t nb, int64_t dps,
    double* __restrict__ part, int nterms) {
  constexpr int R = kGpR, B = kGpBlock, CS = kGpStride;
  constexpr int DS = D <= 2 ? D : (D + 3) / 4 * 4;  // LDS stride of a point
  constexpr int NT = ARD ? D : 1;
  __shared__ __align__(16) float sx[B * DS];
  __shared__ float sl[kGpCols * CS], sr[kGpCols * CS];
  __shared__ double red[4];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lm = lane & 15, lq = lane >> 4;
  const int cn = min(kGpCols, ncols - c0);
  const int csteps = (cn + 3) / 4;
  const int64_t b = blockIdx.x;

  float xi[R][D], lb[R][4], rb[R][4];
#pragma unroll
  for (int r = 0; r < R; ++r) {
    const int64_t i = b * B + (wave * R + r) * 16 + lm;
#pragma unroll
    for (int k = 0; k < D; ++k) xi[r][k] = (i < n && k < d) ? Z[i * d + k] : 0.0f;
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      const int c = 4 * s + lq;
      const bool in = i < n && c < cn;  // points past n carry no weight
      lb[r][s] = in ? Lf[(int64_t)(c0 + c) * n + i] : 0.0f;
      rb[r][s] = in ? Rf[(int64_t)(c0 + c) * n + i] : 0.0f;
    }
  }
  double accd[NT + 1];
#pragma unroll
  for (int t = 0; t <= NT; ++t) accd[t] = 0.0;

  const int64_t d0 = (int64_t)blockIdx.y * dps, d1 = min(d0 + dps, sym_span(b, nb) + 1);
  for (int64_t dl = d0; dl < d1; ++dl) {
    int64_t J = b + dl;
    if (J >= nb) J -= nb;
    const int64_t j0 = J * B;
    const int cnt = (int)min((int64_t)B, n - j0);
    __syncthreads();
    for (int q = threadIdx.x; q < B * D; q += 256) {
      const int jj = q / D, k = q - jj * D;
      sx[jj * DS + k] = (jj < cnt && k < d) ? Z[(j0 + jj) * d + k] : 0.0f;
    }
    for (int q = threadIdx.x; q < B * kGpCols; q += 256) {
      const int c = q / B, jj = q - c * B;
      const bool in = jj < cnt && c < cn;
      sr[c * CS + jj] = in ? Rf[(int64_t)(c0 + c) * n + j0 + jj] : 0.0f;
      sl[c * CS + jj] = in ? Lf[(int64_t)(c0 + c) * n + j0 + jj] : 0.0f;
    }
    __syncthreads();
    const float wt = dl == 0 ? 0.5f : 1.0f;
    const int tiles = (cnt + 15) / 16;
    float acc[NT + 1];
#pragma unroll
    for (int t = 0; t <= NT; ++t) acc[t] = 0.0f;
    auto flush = [&]() __attribute__((always_inline)) {
#pragma unroll
      for (int t = 0; t <= NT; ++t) {
        accd[t] += (double)acc[t];
        acc[t] = 0.0f;
      }
    };
#pragma unroll 1
    for (int ct = 0; ct < tiles; ++ct) {
      f4 wv[R];
#pragma unroll
      for (int r = 0; r < R; ++r) wv[r] = f4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int s = 0; s < 4; ++s) {
        if (s >= csteps) break;
        const float ar = sr[(4 * s + lq) * CS + 16 * ct + lm];
        const float al = sl[(4 * s + lq) * CS + 16 * ct + lm];
#pragma unroll
        for (int r = 0; r < R; ++r) {
          wv[r] = __builtin_amdgcn_mfma_f32_16x16x4f32(ar, lb[r][s], wv[r], 0, 0, 0);
          wv[r] = __builtin_amdgcn_mfma_f32_16x16x4f32(al, rb[r][s], wv[r], 0, 0, 0);
        }
      }
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const float* xp = sx + (16 * ct + 4 * lq + e) * DS;
        float xj[DS];
        if constexpr (D <= 2) {
#pragma unroll
          for (int k = 0; k < D; ++k) xj[k] = xp[k];
        } else {
#pragma unroll
          for (int k = 0; k < DS; k += 4) {
            const f4 x = *reinterpret_cast<const f4*>(xp + k);
#pragma unroll
            for (int q = 0; q < 4; ++q) xj[k + q] = x[q];
          }
        }
#pragma unroll
        for (int r = 0; r < R; ++r) {
          float df[D], r2 = 0.0f;
#pragma unroll
          for (int k = 0; k < D; ++k) {
            df[k] = xi[r][k] - xj[k];
            r2 = fmaf(df[k], df[k], r2);
          }
          float kv, h;
          value_and_h<KIND, ARD>(r2, kv, h);
          const float w = wt * wv[r][e];
          const float hw = h * w;
          acc[NT] = fmaf(kv, w, acc[NT]);
          if constexpr (ARD) {
#pragma unroll
            for (int k = 0; k < D; ++k) acc[k] = fmaf(hw * df[k], df[k], acc[k]);
          } else {
            acc[0] = fmaf(hw, r2, acc[0]);
          }
        }
      }
      if (ct % kGpFlush == kGpFlush - 1) flush();
    }
    flush();
  }
  double* dst = part + ((int64_t)blockIdx.y * gridDim.x + blockIdx.x) * nterms;
#pragma unroll
  for (int t = 0; t <= NT; ++t) {
    double v = accd[t];
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) v += __shfl_xor(v, o);
    __syncthreads();
    if (lane == 0) red[wave] = v;
    __syncthreads();
    const int term = t == NT ? nterms - 1 : t;
    if (threadIdx.x == 0 && (t == NT || t < nterms - 1)) dst[term] = red[0] + red[1] + red[2] + red[3];
  }
}

// acc[q] (+)= sum_b part[b nterms + q]: one wave per term, fixed order.
__global__ __launch_bounds__(64) void k_grad_pair_sum(const double* __restrict__ part,
                                                      int64_t nblk, int nterms, int accumulate,
                                                      double* __restrict__ acc) {
  const int q = blockIdx.x, lane = threadIdx.x;
  double s = 0.0;
#pragma unroll 8
  for (int64_t b = lane; b < nblk; b += 64) s += part[b * nterms + q];
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) s += __shfl_xor(s, o);
  if (lane == 0) acc[q] = accumulate ? acc[q] + s : s;
}

using GpFn = void (*)(const float*, int64_t, int, const float*, const float*, int, int, int64_t,
                      int64_t, double*, int);

// the dimension steps of the difference products (direct.hip)
template <int KIND, bool ARD>
GpFn pick_gp_d(int d) {
#define MGP_GP_CASE(DV) \
  if (d <= DV) return k_grad_pair<KIND, DV, ARD>;
  MGP_GP_CASE(1)
  MGP_GP_CASE(2)
  MGP_GP_CASE(3)
  MGP_GP_CASE(4)
  MGP_GP_CASE(5)
  MGP_GP_CASE(6)
  MGP_GP_CASE(8)
  MGP_GP_CASE(10)
  MGP_GP_CASE(12)
  MGP_GP_CASE(16)
  MGP_GP_CASE(20)
  MGP_GP_CASE(24)
  MGP_GP_CASE(32)
#undef MGP_GP_CASE
  return nullptr;
}

template <int KIND>
GpFn pick_gp_ard(bool ard, int d) {
  return ard ? pick_gp_d<KIND, true>(d) : pick_gp_d<KIND, false>(d);
}

GpFn pick_gp(int kind, bool ard, int d) {
  switch (kind) {
    case KIND_RBF: return pick_gp_ard<KIND_RBF>(ard, d);
    case KIND_MATERN12: return pick_gp_ard<KIND_MATERN12>(ard, d);
    case KIND_MATERN32: return pick_gp_ard<KIND_MATERN32>(ard, d);
    default: return pick_gp_ard<KIND_MATERN52>(ard, d);
  }
}

}  // namespace

void grad_trace_pairs(int kind, bool ard, const PackedPoints& pts, int d, const float* Lf,
                      const float* Rf, int ncols, double* acc_host, GradTraceWorkspace& ws,
                      hipStream_t st) {
  MGP_REQUIRE(d >= 1 && d <= 32, "gradient kernel supports d <= 32");
  const int nterms = ard ? d + 1 : 2;
  const int64_t nb = ceil_div(std::max<int64_t>(pts.n, 1), (int64_t)kGpBlock);
  // one column block a workgroup until that makes 4096 of them
  const int64_t offsets = nb / 2 + 1;
  const int64_t dps = ceil_div(offsets, std::min(offsets, ceil_div(4096, nb)));
  const int64_t splits = ceil_div(offsets, dps);
  const int64_t nblk = nb * splits;
  double* part = ws.part.ensure((size_t)(nblk + 1) * nterms);
  double* acc = part + (size_t)nblk * nterms;
  const GpFn fn = pick_gp(kind, ard, d);
  MGP_REQUIRE(fn != nullptr, "no gradient kernel for this dimension");
  for (int c0 = 0; c0 < ncols; c0 += kGpCols) {
    hipLaunchKernelGGL(fn, dim3((unsigned)nb, (unsigned)splits), dim3(256), 0, st, pts.z.ptr,
                       pts.n, d, Lf, Rf, ncols, c0, nb, dps, part, nterms);
    hipLaunchKernelGGL(k_grad_pair_sum, dim3((unsigned)nterms), dim3(64), 0, st, part, nblk,
                       nterms, c0 > 0 ? 1 : 0, acc);
    MGP_HIP_CHECK(hipGetLastError());
  }
  MGP_HIP_CHECK(hipMemcpyAsync(acc_host, acc, (size_t)nterms * sizeof(double),
                               hipMemcpyDeviceToHost, st));
  MGP_HIP_CHECK(hipStreamSynchronize(st));
}

}  // namespace mgp
