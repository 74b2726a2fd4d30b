// Composite kernel trees on gfx950: products, dense blocks, pivot columns and
// gradient traces evaluated per pair from raw coordinate differences (VALU;
// the Gram-form tile path serves single radial leaves).  Tree semantics and
// reference citations are in kernel_tree.h.
#include "sym_common.h"
#include "tree.h"
#include "tree_jit.h"

#include <algorithm>
#include <cmath>
#include <string>
#include <vector>

namespace mgp {

namespace {

constexpr int kTile = 128;      // column points per LDS tile
constexpr int kMaxCols = 16;    // right-hand sides per pass
constexpr int kGradCols = 16;   // gradient-trace factor columns per pass
typedef float f4t __attribute__((ext_vector_type(4)));
static_assert(kTreeChunk % 4 == 0 && kTile % kTreeChunk == 0, "float4 chunk reads");

void require(bool ok, const std::string& msg) {
  if (!ok) throw Error(ST_INVALID, msg);
}

// out[c][i] = sum_y part[y][c][i] (+ noise V[c][i]), splits summed in order.
__global__ void k_tree_reduce(const float* __restrict__ part, int splits, int64_t m, int ncols,
                              const float* __restrict__ V, float noise, int add_noise,
                              float* __restrict__ out) {
  const int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (idx >= m * ncols) return;
  double s = 0.0;
  for (int y = 0; y < splits; ++y) s += (double)part[(int64_t)y * ncols * m + idx];
  float o = (float)s;
  if (add_noise) o = fmaf(noise, V[idx], o);
  out[idx] = o;
}

// out[c][j] = sum_y fwd[y][c][j] + the transposed partials of the row blocks
// that formed j's column block (delta order) + noise V: fp64, rounded once.
// Four threads per point own four right-hand sides each; unformed slots (nb
// even, the last delta) are read and dropped by a select.
__global__ __launch_bounds__(256) void k_tree_sym_reduce(
    const float* __restrict__ fwd, int splits, const float* __restrict__ tp, int block,
    int64_t nb, int64_t hmax, int64_t n, int nc, float noise, const float* __restrict__ V,
    float* __restrict__ out) {
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
    return __builtin_nontemporal_load(reinterpret_cast<const f4t*>(
        tp + ((bb * hmax + dl - 1) * block + jl) * 16 + c4));
  };
  int64_t dl = 1;
  for (; dl + 8 <= hmax + 1; dl += 8) {
    f4t v[8];
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
    const f4t v = slot(dl, ok);
#pragma unroll
    for (int e = 0; e < 4; ++e) tot[e] += ok ? (double)v[e] : 0.0;
  }
#pragma unroll
  for (int e = 0; e < 4; ++e)
    if (c4 + e < nc) {
      const int64_t idx = (int64_t)(c4 + e) * n + j;
      out[idx] = (float)(tot[e] + (double)noise * (double)V[idx]);
    }
}

// out[i] = K(x_i, x_i)
__global__ void k_tree_self(const float* __restrict__ X, int64_t m, KernelTree t,
                            const float* __restrict__ p, float* __restrict__ out) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= m) return;
  float x[kTreeMaxInputDim];
  for (int k = 0; k < t.d; ++k) x[k] = X[i * t.d + k];
  out[i] = tree_value(t, p, x, x);
}

// out[c*n + i] = K(rows[r0 + c], cols[i])
__global__ void k_tree_fill(const float* __restrict__ Xr, int64_t r0, int64_t rows,
                            const float* __restrict__ Xc, int64_t n, KernelTree t,
                            const float* __restrict__ p, float* __restrict__ out) {
  const int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (idx >= rows * n) return;
  const int64_t c = idx / n, i = idx - c * n;
  const int d = t.d;
  float xr[kTreeMaxInputDim], xc[kTreeMaxInputDim];
  for (int k = 0; k < d; ++k) {
    xr[k] = Xr[(r0 + c) * d + k];
    xc[k] = Xc[i * d + k];
  }
  out[idx] = tree_value(t, p, xr, xc);
}

// part[(y*gx + x)*P + q] = sum over the block's pairs (a, b) of
// dK_ab/dtheta_q sum_c Lf[c][a] Rf[c][b]; grid = (row blocks, column splits).
__global__ __launch_bounds__(256) void k_tree_grad_trace(
    const float* __restrict__ X, int64_t n, KernelTree t, const float* __restrict__ p,
    const float* __restrict__ Lf, const float* __restrict__ Rf, int ncols, int c0,
    double* __restrict__ part) {
  __shared__ float xb[64][kTreeMaxInputDim];
  __shared__ float rb[64][kGradCols];
  __shared__ double red[256];
  const int d = t.d, P = t.nparams;
  const int cn = min(kGradCols, ncols - c0);
  const int64_t a = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const bool live = a < n;
  float xa[kTreeMaxInputDim], la[kGradCols];
  for (int k = 0; k < d; ++k) xa[k] = live ? X[a * d + k] : 0.0f;
  for (int c = 0; c < kGradCols; ++c) la[c] = (live && c < cn) ? Lf[(int64_t)(c0 + c) * n + a] : 0.0f;
  const int64_t tiles = (n + 63) / 64;
  const int64_t tps = (tiles + gridDim.y - 1) / gridDim.y;
  const int64_t jb = min(n, (int64_t)blockIdx.y * tps * 64);
  const int64_t je = min(n, jb + tps * 64);
  double accd[kTreeMaxParams];
  for (int q = 0; q < kTreeMaxParams; ++q) accd[q] = 0.0;
  for (int64_t b0 = jb; b0 < je; b0 += 64) {
    __syncthreads();
    for (int q = threadIdx.x; q < 64 * kTreeMaxInputDim; q += blockDim.x) {
      const int bb = q / kTreeMaxInputDim, k = q - bb * kTreeMaxInputDim;
      const int64_t b = b0 + bb;
      xb[bb][k] = (b < je && k < d) ? X[b * d + k] : 0.0f;
    }
    for (int q = threadIdx.x; q < 64 * kGradCols; q += blockDim.x) {
      const int bb = q / kGradCols, c = q - bb * kGradCols;
      const int64_t b = b0 + bb;
      rb[bb][c] = (b < je && c < cn) ? Rf[(int64_t)(c0 + c) * n + b] : 0.0f;
    }
    __syncthreads();
    float g[kTreeMaxParams];
    for (int q = 0; q < kTreeMaxParams; ++q) g[q] = 0.0f;
    const int cnt = (int)min((int64_t)64, je - b0);
    if (live) {
      for (int bb = 0; bb < cnt; ++bb) {
        float w = 0.0f;
        for (int c = 0; c < kGradCols; ++c) w = fmaf(la[c], rb[bb][c], w);
        tree_grad_accumulate(t, p, xa, xb[bb], w, g);
      }
    }
    for (int q = 0; q < P; ++q) accd[q] += (double)g[q];
  }
  for (int q = 0; q < P; ++q) {
    red[threadIdx.x] = live ? accd[q] : 0.0;
    __syncthreads();
    for (int s = blockDim.x / 2; s > 0; s >>= 1) {
      if ((int)threadIdx.x < s) red[threadIdx.x] += red[threadIdx.x + s];
      __syncthreads();
    }
    if (threadIdx.x == 0) part[((int64_t)blockIdx.y * gridDim.x + blockIdx.x) * P + q] = red[0];
    __syncthreads();
  }
}

// part[(y*gx + x)*table_size + e] = sum over the block's pairs (a, b) of
// w_ab dK_ab/dv_l at table entry e = p0_l + level_a * L + level_b of every
// categorical leaf l, with w_ab = sum_c Lf[c][a] Rf[c][b].
__global__ __launch_bounds__(256) void k_tree_cat_grad(
    const float* __restrict__ X, int64_t n, KernelTree t, const float* __restrict__ p,
    const float* __restrict__ Lf, const float* __restrict__ Rf, int ncols, int c0,
    double* __restrict__ part) {
  __shared__ float xb[64][kTreeMaxInputDim];
  __shared__ float rb[64][kGradCols];
  __shared__ float tab[kTreeMaxTable];
  const int d = t.d;
  const int cn = min(kGradCols, ncols - c0);
  const int64_t a = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const bool live = a < n;
  for (int e = threadIdx.x; e < t.table_size; e += blockDim.x) tab[e] = 0.0f;
  float xa[kTreeMaxInputDim], la[kGradCols];
  for (int k = 0; k < d; ++k) xa[k] = live ? X[a * d + k] : 0.0f;
  for (int c = 0; c < kGradCols; ++c) la[c] = (live && c < cn) ? Lf[(int64_t)(c0 + c) * n + a] : 0.0f;
  float acc[kTreeMaxCatRow];
  for (int q = 0; q < kTreeMaxCatRow; ++q) acc[q] = 0.0f;
  const int64_t tiles = (n + 63) / 64;
  const int64_t tps = (tiles + gridDim.y - 1) / gridDim.y;
  const int64_t jb = min(n, (int64_t)blockIdx.y * tps * 64);
  const int64_t je = min(n, jb + tps * 64);
  for (int64_t b0 = jb; b0 < je; b0 += 64) {
    __syncthreads();
    for (int q = threadIdx.x; q < 64 * kTreeMaxInputDim; q += blockDim.x) {
      const int bb = q / kTreeMaxInputDim, k = q - bb * kTreeMaxInputDim;
      const int64_t b = b0 + bb;
      xb[bb][k] = (b < je && k < d) ? X[b * d + k] : 0.0f;
    }
    for (int q = threadIdx.x; q < 64 * kGradCols; q += blockDim.x) {
      const int bb = q / kGradCols, c = q - bb * kGradCols;
      const int64_t b = b0 + bb;
      rb[bb][c] = (b < je && c < cn) ? Rf[(int64_t)(c0 + c) * n + b] : 0.0f;
    }
    __syncthreads();
    const int cnt = (int)min((int64_t)64, je - b0);
    if (live) {
      for (int bb = 0; bb < cnt; ++bb) {
        float w = 0.0f;
        for (int c = 0; c < kGradCols; ++c) w = fmaf(la[c], rb[bb][c], w);
        float ladj[kTreeMaxLeaves];
        tree_leaf_adjoints(t, p, xa, xb[bb], w, ladj);
        int off = 0;
        for (int l = 0; l < t.nleaves; ++l) {
          const TreeLeaf& lf = t.leaf[l];
          if (lf.kind != KIND_CAT) continue;
          acc[off + tree_level(xb[bb][t.dims[lf.dim_off]], lf.ard)] += ladj[l];
          off += lf.ard;
        }
      }
    }
  }
  __syncthreads();
  if (live) {
    int off = 0;
    for (int l = 0; l < t.nleaves; ++l) {
      const TreeLeaf& lf = t.leaf[l];
      if (lf.kind != KIND_CAT) continue;
      const int L = lf.ard;
      const int row = lf.p0 + tree_level(xa[t.dims[lf.dim_off]], L) * L;
      for (int lb = 0; lb < L; ++lb) atomicAdd(&tab[row + lb], acc[off + lb]);
      off += L;
    }
  }
  __syncthreads();
  double* dst = part + ((int64_t)blockIdx.y * gridDim.x + blockIdx.x) * t.table_size;
  for (int e = threadIdx.x; e < t.table_size; e += blockDim.x) dst[e] = (double)tab[e];
}

}  // namespace

KernelTree parse_kernel_tree(const int* spec, int len) {
  require(spec != nullptr && len >= 4, "kernel tree spec is too short");
  KernelTree t;
  int pos = 0;
  auto next = [&]() {
    require(pos < len, "kernel tree spec is truncated");
    return spec[pos++];
  };
  t.d = next();
  t.nparams = next();
  t.nleaves = next();
  t.nnodes = next();
  require(t.d >= 1 && t.d <= kTreeMaxInputDim, "kernel tree input dimension must be in [1, 32]");
  require(t.nparams >= 1 && t.nparams <= kTreeMaxParams, "kernel tree has too many parameters");
  require(t.nleaves >= 1 && t.nleaves <= kTreeMaxLeaves, "kernel tree needs 1..8 leaves");
  require(t.nnodes >= 1 && t.nnodes <= kTreeMaxNodes, "kernel tree needs 1..16 nodes");
  int doff = 0, cat_levels = 0;
  for (int l = 0; l < t.nleaves; ++l) {
    TreeLeaf& lf = t.leaf[l];
    lf.kind = next();
    lf.ard = next();
    lf.ndim = next();
    lf.p0 = next();
    lf.dim_off = doff;
    lf.deg = 0;
    if (lf.kind == KIND_POLY) {
      lf.deg = next();
      require(lf.deg >= 1 && lf.deg <= 16, "polynomial degree must be an integer in [1, 16]");
    }
    require(lf.kind >= KIND_RBF && lf.kind <= KIND_POLY, "unknown kernel tree leaf kind");
    require(lf.ndim >= 1 && doff + lf.ndim <= kTreeMaxDims, "kernel tree leaf dimensions");
    for (int q = 0; q < lf.ndim; ++q) {
      const int dq = next();
      require(dq >= 0 && dq < t.d, "kernel tree leaf dimension out of range");
      t.dims[doff++] = dq;
    }
    if (lf.kind == KIND_CAT) {
      require(lf.ndim == 1, "a categorical leaf reads one input column");
      require(lf.ard >= 2 && lf.ard <= kTreeMaxLevels, "categorical leaves need 2..32 levels");
      require(lf.p0 >= 0 && lf.p0 + lf.ard * lf.ard <= kTreeMaxTable,
              "categorical tables exceed 1024 entries");
      t.table_size = std::max(t.table_size, lf.p0 + lf.ard * lf.ard);
      t.ncat += 1;
      cat_levels += lf.ard;
      continue;
    }
    const int nls = lf.ard ? lf.ndim : 1;
    const int extra = (lf.kind == KIND_RQ || lf.kind == KIND_PERIODIC) ? 1
                      : lf.kind == KIND_POLY                           ? 2
                                                                       : 0;
    require(lf.p0 >= 0 && lf.p0 + nls + extra + 1 <= t.nparams,
            "kernel tree leaf parameters out of range");
    if (lf.kind == KIND_LINEAR || lf.kind == KIND_POLY) t.nonstationary = 1;
  }
  require(cat_levels <= kTreeMaxCatRow, "categorical leaves exceed 64 levels in total");
  int leaf_uses[kTreeMaxLeaves] = {0};
  for (int i = 0; i < t.nnodes; ++i) {
    TreeNode& nd = t.node[i];
    nd.code = next();
    nd.a = next();
    nd.b = next();
    switch (nd.code) {
      case TN_LEAF:
        require(nd.a >= 0 && nd.a < t.nleaves, "kernel tree leaf node index");
        require(++leaf_uses[nd.a] == 1, "a kernel tree leaf appears in more than one node");
        break;
      case TN_ADD:
      case TN_MUL:
        require(nd.a >= 0 && nd.a < i && nd.b >= 0 && nd.b < i, "kernel tree child order");
        break;
      case TN_SCALE:
        require(nd.a >= 0 && nd.a < i, "kernel tree child order");
        require(nd.b >= 0 && nd.b < t.nparams, "kernel tree scale parameter index");
        break;
      default:
        require(false, "unknown kernel tree node code");
    }
  }
  require(pos == len, "kernel tree spec has trailing entries");
  for (int l = 0; l < t.nleaves; ++l)
    require(leaf_uses[l] == 1, "every kernel tree leaf needs one leaf node");
  return t;
}

double tree_diag(const KernelTree& t, const float* params) {
  std::vector<double> v((size_t)t.nnodes);
  for (int i = 0; i < t.nnodes; ++i) {
    const TreeNode& nd = t.node[i];
    if (nd.code == TN_LEAF && t.leaf[nd.a].kind == KIND_CAT) {
      v[i] = 1.0;  // every correlation table has a unit diagonal
    } else if (nd.code == TN_LEAF) {
      const TreeLeaf& lf = t.leaf[nd.a];
      const int nls = lf.ard ? lf.ndim : 1;
      const int extra = (lf.kind == KIND_RQ || lf.kind == KIND_PERIODIC) ? 1
                        : lf.kind == KIND_POLY                           ? 2
                                                                         : 0;
      // os of a stationary leaf at zero distance (linear / polynomial trees
      // take per-point diagonals, tree_self_values)
      v[i] = (double)params[lf.p0 + nls + extra];
    } else if (nd.code == TN_ADD) {
      v[i] = v[(size_t)nd.a] + v[(size_t)nd.b];
    } else if (nd.code == TN_MUL) {
      v[i] = v[(size_t)nd.a] * v[(size_t)nd.b];
    } else {
      v[i] = (double)params[nd.b] * v[(size_t)nd.a];
    }
  }
  return v[(size_t)t.nnodes - 1];
}

namespace {
// Cost of one pair's value in units of a dimension's part of it: a leaf's
// exponential and the like weigh about five.
int tree_cost(const KernelTree& t) {
  int c = 0;
  for (int l = 0; l < t.nleaves; ++l) c += 5 + t.leaf[l].ndim;
  return c;
}

// Square products with 5 to 16 right-hand sides run on the symmetric kernel
// where n + 100 tree_cost >= 8600 (and n >= 5000, the smallest size at which a
// costly tree gained clearly): below, the blocks fill too few rounds of the
// chip, the dearer a value the earlier half of them pays (11 columns, one-sided
// / symmetric us: RQ in 1 dimension, cost 6, n = 7500 77 / 75, 8000 85 / 74,
// 16000 206 / 173; RBF + Matern-5/2 in 1, cost 12, 7000 95 / 89, 8000 113 / 92;
// RBF x periodic + RQ in 4, cost 24, 5500 83 / 81, 6000 89 / 87, 6500 102 / 88,
// 20000 600 / 458; four leaves in 4, cost 33, 5000 103 / 85).
// Compilation takes 0.14 s the first time (later processes read the runtime's
// disk cache, ~5 ms), in place of the one-sided kernels' 0.21 s for a fit (11
// columns throughout), beside it once predictions need those too; a fit of 100
// steps of up to 100 iterations saves that from about this line on.
constexpr int64_t kTreeSymMin = 5000, kTreeSymBase = 8600, kTreeSymPerCost = 100;
constexpr int kTreeSymMinCols = 5;
constexpr double kTreeSymMaxBytes = 8e9;

// out = (K + noise I) V for nc <= 16 columns on the symmetric kernel.  False,
// with nothing launched, where its partial sums do not fit the device.
bool tree_sym_matvec(const KernelTree& t, const float* p_dev, const float* X, int64_t n,
                     const float* V, int nc, float noise, float* out, DevBuf<float>& work,
                     hipStream_t st) {
  const TreeSymJitKernel jk = tree_sym_jit_kernel(t);
  int dev = 0, cus = 0;
  MGP_HIP_CHECK(hipGetDevice(&dev));
  MGP_HIP_CHECK(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev));
  const int64_t nb = ceil_div(n, (int64_t)jk.block), hmax = nb / 2;
  const int64_t stages = (hmax + 1) * (jk.block / jk.stage);
  const int64_t slots = (int64_t)std::max(cus, 1) * jk.per_cu;
  // rounds of (stages a workgroup + about a third of one of set-up); a split's
  // forward partials cost little beside a stage
  int64_t best = 1;
  double best_cost = 0.0;
  for (int64_t s = 1; s <= std::min<int64_t>(stages, 64); ++s) {
    const int64_t sps = ceil_div(stages, s);
    if (ceil_div(stages, sps) != s) continue;
    const double cost = (double)ceil_div(nb * s, slots) * ((double)sps + 0.35) + 0.02 * (double)s;
    if (s == 1 || cost < best_cost) {
      best_cost = cost;
      best = s;
    }
  }
  long long nn = n, nbb = nb, sp = best, sps = ceil_div(stages, best), hm = hmax;
  const size_t nf = (size_t)best * 16 * nb * jk.block;
  float* fwd = work.try_ensure(nf + (size_t)std::max<int64_t>(nb * hmax, 1) * jk.block * 16);
  if (fwd == nullptr) return false;
  float* tp = fwd + nf;
  int ncc = nc;
  void* args[] = {(void*)&X, &nn, (void*)&p_dev, (void*)&V, &ncc, &nbb, &sp, &sps, &hm,
                  (void*)&fwd, (void*)&tp};
  MGP_HIP_CHECK(hipModuleLaunchKernel(jk.fn, (unsigned)nb, (unsigned)best, 1, 256, 1, 1, 0, st,
                                      args, nullptr));
  hipLaunchKernelGGL(k_tree_sym_reduce, dim3((unsigned)ceil_div(4 * n, 256)), dim3(256), 0, st, fwd,
                     (int)best, tp, jk.block, nb, hmax, n, nc, noise, V, out);
  MGP_HIP_CHECK(hipGetLastError());
  return true;
}

bool tree_sym_route(const KernelTree& t, int64_t m, int64_t n, int nc, bool square) {
  if (!square || m != n || t.table_size != 0) return false;
  if ((double)n * (double)n * 16 * 4 / 512 > kTreeSymMaxBytes) return false;
  const int mode = sym_switch();
  if (mode >= 0) return mode == 1;
  return n >= kTreeSymMin && n + kTreeSymPerCost * tree_cost(t) >= kTreeSymBase &&
         nc >= kTreeSymMinCols;
}
}  // namespace

void tree_matvec(const KernelTree& t, const float* p_dev, const float* Xr, int64_t m,
                 const float* Xc, int64_t n, const float* V, int ncols, float noise,
                 bool square, float* out, DevBuf<float>& work, hipStream_t st) {
  if (m <= 0) return;
  // Column splits so that the launch covers the chip (>= ~2048 blocks of
  // 256 rows), at least one 128-column tile per split.
  const int64_t rows = ceil_div(m, 256);
  const int64_t tiles = ceil_div(std::max<int64_t>(n, 1), kTile);
  const int splits = (int)std::max<int64_t>(
      1, std::min<int64_t>(ceil_div(2048, rows), tiles));
  for (int c0 = 0; c0 < ncols; c0 += kMaxCols) {
    const int nc = std::min(kMaxCols, ncols - c0);
    if (Xr == Xc && tree_sym_route(t, m, n, nc, square) &&
        tree_sym_matvec(t, p_dev, Xc, n, V + (int64_t)c0 * n, nc, noise, out + (int64_t)c0 * n,
                        work, st))
      continue;
    float* part = work.ensure((size_t)splits * nc * m);
    // the tree's straight-line kernel (tree_jit.hip)
    const TreeJitKernel jk = tree_jit_kernel(t, nc);
    const int64_t rblocks = ceil_div(m, jk.rows_per_block);
    {
      const float* vc = V + (int64_t)c0 * n;
      long long mm = m, nn = n;
      int ncc = nc;
      void* args[] = {(void*)&Xr, &mm, (void*)&Xc, &nn, (void*)&p_dev, (void*)&vc, &ncc,
                      (void*)&part};
      MGP_HIP_CHECK(hipModuleLaunchKernel(jk.fn, (unsigned)rblocks, (unsigned)splits, 1, 256, 1, 1,
                                          (unsigned)jk.lds_bytes, st, args, nullptr));
    }
    hipLaunchKernelGGL(k_tree_reduce, dim3((unsigned)ceil_div(m * nc, 256)), dim3(256), 0, st,
                       part, splits, m, nc, V + (int64_t)c0 * n, noise, square ? 1 : 0,
                       out + (int64_t)c0 * m);
    MGP_HIP_CHECK(hipGetLastError());
  }
}

void tree_self_values(const KernelTree& t, const float* p_dev, const float* X, int64_t m,
                      float* out, hipStream_t st) {
  if (m <= 0) return;
  hipLaunchKernelGGL(k_tree_self, dim3((unsigned)ceil_div(m, 256)), dim3(256), 0, st, X, m, t,
                     p_dev, out);
  MGP_HIP_CHECK(hipGetLastError());
}

void tree_fill(const KernelTree& t, const float* p_dev, const float* Xr, int64_t r0,
               int64_t rows, const float* Xc, int64_t n, float* out, hipStream_t st) {
  const int64_t total = rows * n;
  if (total == 0) return;
  hipLaunchKernelGGL(k_tree_fill, dim3((unsigned)ceil_div(total, 256)), dim3(256), 0, st, Xr,
                     r0, rows, Xc, n, t, p_dev, out);
  MGP_HIP_CHECK(hipGetLastError());
}

namespace {
// acc[q] (+)= sum_b part[b * Q + q] for q < Q: one wave per q, lane l sums
// b = l, l + 64, .. in order, then a butterfly of shuffles (fixed order).
__global__ void k_tree_part_sum(const double* __restrict__ part, int64_t nblk, int Q,
                                int accumulate, double* __restrict__ acc) {
  const int q = blockIdx.x, lane = threadIdx.x;
  double s = 0.0;
  for (int64_t b = lane; b < nblk; b += 64) s += part[b * Q + q];
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) s += __shfl_xor(s, o);
  if (lane == 0) acc[q] = accumulate ? acc[q] + s : s;
}

// Column splits of the interpreted traces: one 64-column LDS tile at least
// (a pair takes a thread ~6 us, so small models need the blocks: 6.5 -> 0.5
// ms at n = 1000 against 1024 columns a split).
int64_t grad_splits(int64_t n) {
  const int64_t rows = ceil_div(n, 256);
  return std::max<int64_t>(1, std::min<int64_t>(ceil_div(2048, rows), ceil_div(n, 64)));
}

// The trace runs on the tree's generated kernel where n^2 tree_cost reaches
// this: its compilation takes 0.15 s the first time, and a trace is
// ~0.165 ms (n / 10000)^2 tree_cost shorter than the interpreted one, so from
// here on a fit of 100 steps (the default) in a fresh process repays it (11
// factor columns, interpreted / generated ms: RQ in 1 dimension, cost 6, n =
// 12000 1.48 / 0.18; RBF + Matern-5/2 in 1, cost 12, 8000 1.27 / 0.13, 9000 1.67
// / 0.15; RBF x periodic + RQ in 4, cost 24, 6000 1.90 / 0.13, 10000 4.41 /
// 0.22; four leaves in 4, cost 33, 5000 1.62 / 0.14).  Below, and for trees
// whose leaves share parameter slots, the interpreted kernel.
constexpr double kTreeGradJitWork = 9e8;
}  // namespace

void tree_cat_grad_tables(const KernelTree& t, const float* p_dev, const float* X, int64_t n,
                          const float* Lf, const float* Rf, int ncols, double* G_host,
                          DevBuf<double>& work, hipStream_t st) {
  const int S = t.table_size;
  for (int e = 0; e < S; ++e) G_host[e] = 0.0;
  if (S == 0) return;
  const int64_t rows = ceil_div(n, 256), splits = grad_splits(n), nblk = rows * splits;
  double* part = work.ensure((size_t)nblk * S + S);
  double* acc = part + (size_t)nblk * S;
  for (int c0 = 0; c0 < ncols; c0 += kGradCols) {
    hipLaunchKernelGGL(k_tree_cat_grad, dim3((unsigned)rows, (unsigned)splits), dim3(256), 0, st,
                       X, n, t, p_dev, Lf, Rf, ncols, c0, part);
    hipLaunchKernelGGL(k_tree_part_sum, dim3((unsigned)S), dim3(64), 0, st, part, nblk, S,
                       c0 > 0 ? 1 : 0, acc);
    MGP_HIP_CHECK(hipGetLastError());
  }
  MGP_HIP_CHECK(hipMemcpyAsync(G_host, acc, (size_t)S * sizeof(double), hipMemcpyDeviceToHost,
                               st));
  MGP_HIP_CHECK(hipStreamSynchronize(st));
}

void tree_grad_traces(const KernelTree& t, const float* p_dev, const float* X, int64_t n,
                      const float* Lf, const float* Rf, int ncols, double* g_host,
                      DevBuf<double>& work, hipStream_t st) {
  const int P = t.nparams;
  TreeGradJitKernel jk;
  if ((double)n * (double)n * tree_cost(t) >= kTreeGradJitWork) jk = tree_grad_jit_kernel(t);
  int64_t rows = ceil_div(n, 256), splits = grad_splits(n), dps = 0;
  if (jk.fn) {
    rows = ceil_div(n, (int64_t)jk.block);
    const int64_t offsets = jk.symmetric ? rows / 2 + 1 : rows;
    dps = ceil_div(offsets, std::min(offsets, ceil_div(4096, rows)));
    splits = ceil_div(offsets, dps);
  }
  const int64_t nblk = rows * splits;
  double* part = work.ensure((size_t)nblk * P + P);
  double* acc = part + (size_t)nblk * P;
  for (int c0 = 0; c0 < ncols; c0 += kGradCols) {
    if (jk.fn) {
      long long nn = n, nb = rows, dd = dps;
      int nc = ncols, cc = c0;
      void* args[] = {(void*)&X,  &nn, (void*)&p_dev, (void*)&Lf, (void*)&Rf, &nc, &cc,
                      &nb, &dd, (void*)&part};
      MGP_HIP_CHECK(hipModuleLaunchKernel(jk.fn, (unsigned)rows, (unsigned)splits, 1, 256, 1, 1, 0,
                                          st, args, nullptr));
    } else {
      hipLaunchKernelGGL(k_tree_grad_trace, dim3((unsigned)rows, (unsigned)splits), dim3(256), 0,
                         st, X, n, t, p_dev, Lf, Rf, ncols, c0, part);
    }
    hipLaunchKernelGGL(k_tree_part_sum, dim3((unsigned)P), dim3(64), 0, st, part, nblk, P,
                       c0 > 0 ? 1 : 0, acc);
    MGP_HIP_CHECK(hipGetLastError());
  }
  MGP_HIP_CHECK(hipMemcpyAsync(g_host, acc, (size_t)P * sizeof(double), hipMemcpyDeviceToHost,
                               st));
  MGP_HIP_CHECK(hipStreamSynchronize(st));
}

}  // namespace mgp
