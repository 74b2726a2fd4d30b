// Straight-line product kernels of composite kernel trees, compiled at run time
// with hiprtc: the gfx950 counterpart of the reference's per-kernel code
// generation (codegen_engine/emit/gpu_kernel.py:151-260 emits one Mojo kernel
// per kernel expression; expressions.py:77-421 holds the leaf formulas).
//
// The interpreted tree kernels (tree.hip) walk the node list per pair with the
// node values in private memory.  Here the tree's value is emitted as one
// expression per leaf and node, with the leaf constants (inverse
// lengthscales, outputscales, ...) computed once per thread from the
// parameter vector, so a pair costs only its arithmetic: coordinates come
// from broadcast LDS reads, the products accumulate in registers.  The leaf
// arithmetic is the interpreted chunk evaluator's (kernel_tree.h,
// tree_leaf_chunk), term for term.  One compile per (tree, device), cached
// for the process.
#include "tree_jit.h"

#include <hip/hiprtc.h>

#include <map>
#include <mutex>
#include <sstream>
#include <string>
#include <tuple>
#include <vector>

namespace mgp {

namespace {

constexpr int kJitTile = 128;  // column points per LDS tile
const int kJitCols[] = {1, 2, 4, 8, 16};
constexpr int kJitMfmaMinCols = 8;   // column counts from here use the MFMA product
constexpr int kJitMfmaRowTiles = 2;  // 16-row tiles per wave in the MFMA kernel
constexpr int kTreeSymBlock = 256;   // points per block of the symmetric product kernel
constexpr int kTreeSymStage = 64;    // columns per LDS stage of it
constexpr int kTreeGradBlock = 128;  // points per block of the gradient kernel

std::string f(float v) {
  std::ostringstream o;
  o.precision(9);
  o << std::scientific << v << "f";
  return o.str();
}

// Prologue (per-thread constants from p) and pair code (from xi, xj) of the
// tree; leaf l's value is l<l>, node i's n<i>, the tree value the last node's.
// The per-dimension terms and exponentials keep names of their own for the
// gradient code below.
void emit_tree(const KernelTree& t, std::string& pro, std::string& pair) {
  std::ostringstream P, Q;
  for (int l = 0; l < t.nleaves; ++l) {
    const TreeLeaf& lf = t.leaf[l];
    const int nls = lf.ard ? lf.ndim : 1;
    const std::string L = "l" + std::to_string(l);
    auto dim = [&](int q) { return t.dims[lf.dim_off + q]; };
    if (lf.kind == KIND_CAT) {
      const int L_ = lf.ard;
      Q << "  float " << L << ";\n  {\n"
        << "    int a = (int)xi[" << dim(0) << "], b = (int)xj[" << dim(0) << "];\n"
        << "    a = a < 0 ? 0 : (a >= " << L_ << " ? " << L_ - 1 << " : a);\n"
        << "    b = b < 0 ? 0 : (b >= " << L_ << " ? " << L_ - 1 << " : b);\n"
        << "    " << L << " = p[" << t.nparams + lf.p0 << " + a * " << L_ << " + b];\n  }\n";
      continue;
    }
    if (lf.kind == KIND_LINEAR || lf.kind == KIND_POLY) {
      for (int q = 0; q < nls; ++q)
        P << "  const float " << L << "w" << q << " = p[" << lf.p0 + q << "];\n";
      P << "  const float " << L << "os = p[" << lf.p0 + nls + (lf.kind == KIND_POLY ? 2 : 0)
        << "];\n";
      if (lf.kind == KIND_POLY)
        P << "  const float " << L << "off = p[" << lf.p0 + nls + 1 << "];\n";
      Q << "  float " << L << "d = 0.0f;\n";
      for (int q = 0; q < lf.ndim; ++q) {
        const std::string xx = L + "x" + std::to_string(q);
        Q << "  const float " << xx << " = xi[" << dim(q) << "] * xj[" << dim(q) << "];\n";
        if (lf.ard)
          Q << "  " << L << "d = fmaf(" << L << "w" << q << ", " << xx << ", " << L << "d);\n";
        else
          Q << "  " << L << "d = " << L << "d + " << xx << ";\n";
      }
      if (!lf.ard)
        Q << "  const float " << L << "raw = " << L << "d;\n  " << L << "d *= " << L << "w0;\n";
      if (lf.kind == KIND_LINEAR) {
        Q << "  const float " << L << " = " << L << "os * " << L << "d;\n";
      } else {
        Q << "  const float " << L << "B = " << L << "d + " << L << "off;\n"
          << "  float " << L << "bp = 1.0f;\n";
        for (int k = 1; k < lf.deg; ++k) Q << "  " << L << "bp *= " << L << "B;\n";
        Q << "  const float " << L << " = " << L << "os * " << L << "bp * " << L << "B;\n";
      }
      continue;
    }
    // radial, RQ and periodic leaves: inverse lengthscales
    for (int q = 0; q < nls; ++q)
      P << "  const float " << L << "il" << q << " = 1.0f / p[" << lf.p0 + q << "];\n";
    if (lf.kind == KIND_PERIODIC) {
      P << "  const float " << L << "ip = " << f(kTreePi) << " / p[" << lf.p0 + nls << "];\n"
        << "  const float " << L << "os = p[" << lf.p0 + nls + 1 << "];\n";
      Q << "  float " << L << "s = 0.0f;\n";
      for (int q = 0; q < lf.ndim; ++q)
        Q << "  const float " << L << "t" << q << " = (xi[" << dim(q) << "] - xj[" << dim(q)
          << "]) * " << L << "ip, " << L << "n" << q << " = __sinf(" << L << "t" << q << ");\n  "
          << L << "s = fmaf(" << L << "n" << q << " * " << L << "n" << q << ", " << L << "il"
          << (lf.ard ? q : 0) << ", " << L << "s);\n";
      Q << "  const float " << L << " = " << L << "os * __expf(-2.0f * " << L << "s);\n";
      continue;
    }
    Q << "  float " << L << "r2 = 0.0f;\n";
    for (int q = 0; q < lf.ndim; ++q)
      Q << "  const float " << L << "u" << q << " = (xi[" << dim(q) << "] - xj[" << dim(q)
        << "]) * " << L << "il" << (lf.ard ? q : 0) << "; " << L << "r2 = fmaf(" << L << "u" << q
        << ", " << L << "u" << q << ", " << L << "r2);\n";
    if (lf.kind == KIND_RQ) {
      P << "  const float " << L << "al = p[" << lf.p0 + nls << "];\n"
        << "  const float " << L << "ia = 0.5f / " << L << "al;\n"
        << "  const float " << L << "os = p[" << lf.p0 + nls + 1 << "];\n";
      Q << "  const float " << L << "B = fmaf(" << L << "r2, " << L << "ia, 1.0f), " << L
        << "lb = __log2f(" << L << "B);\n"
        << "  const float " << L << " = " << L << "os * exp2f(-" << L << "al * " << L << "lb);\n";
      continue;
    }
    P << "  const float " << L << "os = p[" << lf.p0 + nls << "];\n";
    if (lf.kind == KIND_RBF) {
      Q << "  const float " << L << " = " << L << "os * __expf(-0.5f * " << L << "r2);\n";
      continue;
    }
    Q << "  const float " << L << "r = sqrtf(fmaxf(" << L << "r2 + 1e-20f, 1e-20f));\n";
    if (lf.kind == KIND_MATERN12) {
      // the -20 clamp applies to ARD Matern-1/2 leaves only (exp2_limit)
      if (lf.ard)
        Q << "  const float " << L << " = " << L << "os * __expf(fmaxf(-" << L
          << "r, -20.0f));\n";
      else
        Q << "  const float " << L << " = " << L << "os * __expf(-" << L << "r);\n";
    } else if (lf.kind == KIND_MATERN32) {
      Q << "  const float " << L << "s3 = 1.7320508075688772f * " << L << "r;\n"
        << "  const float " << L << "e = __expf(fmaxf(-" << L << "s3, -20.0f));\n"
        << "  const float " << L << " = " << L << "os * (1.0f + " << L << "s3) * " << L << "e;\n";
    } else {
      Q << "  const float " << L << "s5 = 2.2360679774997897f * " << L << "r;\n"
        << "  const float " << L << "e = __expf(fmaxf(-" << L << "s5, -20.0f));\n"
        << "  const float " << L << " = " << L << "os * (1.0f + " << L << "s5 + (5.0f / 3.0f) * "
        << L << "r2) * " << L << "e;\n";
    }
  }
  for (int i = 0; i < t.nnodes; ++i) {
    const TreeNode& nd = t.node[i];
    const std::string N = "n" + std::to_string(i);
    if (nd.code == TN_LEAF)
      Q << "  const float " << N << " = l" << nd.a << ";\n";
    else if (nd.code == TN_ADD)
      Q << "  const float " << N << " = n" << nd.a << " + n" << nd.b << ";\n";
    else if (nd.code == TN_MUL)
      Q << "  const float " << N << " = n" << nd.a << " * n" << nd.b << ";\n";
    else {
      P << "  const float s" << i << " = p[" << nd.b << "];\n";
      Q << "  const float " << N << " = s" << i << " * n" << nd.a << ";\n";
    }
  }
  pro = P.str();
  pair = Q.str();
}
std::string tree_value_return(const KernelTree& t) {
  return "  return n" + std::to_string(t.nnodes - 1) + ";\n";
}

// The kernel source: out partials part[y][c][i] = sum over split y of
// K(Xr_i, Xc_j) V[c][j] for c < nc (the interpreted kernel's layout), one row
// per thread, NC >= nc accumulators.
std::string tree_source(const KernelTree& t) {
  std::string pro, pair;
  emit_tree(t, pro, pair);
  pair += tree_value_return(t);
  const int D = t.d, DP = (D + 3) / 4 * 4;
  std::ostringstream s;
  s << "#define D " << D << "\n#define DP " << DP << "\n#define TILE " << kJitTile << "\n"
    << "template <int NC>\n"
    << "__device__ __forceinline__ void body(const float* __restrict__ Xr, long long m,\n"
    << "    const float* __restrict__ Xc, long long n, const float* __restrict__ p,\n"
    << "    const float* __restrict__ V, int nc, float* __restrict__ part) {\n"
    << "  extern __shared__ float sm[];\n"
    << "  float* sx = sm;\n"
    << "  float* sv = sm + TILE * DP;\n"
    << pro
    << "  auto kval = [&](const float* __restrict__ xi, const float* __restrict__ xj)\n"
    << "      __attribute__((always_inline)) -> float {\n"
    << pair
    << "  };\n"
    << "  const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;\n"
    << "  float xi[DP];\n"
    << "#pragma unroll\n"
    << "  for (int k = 0; k < DP; ++k) xi[k] = (i < m && k < D) ? Xr[i * D + k] : 0.0f;\n"
    << "  double acc[NC];\n"
    << "#pragma unroll\n"
    << "  for (int c = 0; c < NC; ++c) acc[c] = 0.0;\n"
    << "  const long long tiles = (n + TILE - 1) / TILE;\n"
    << "  const long long tps = (tiles + gridDim.y - 1) / gridDim.y;\n"
    << "  const long long jbeg = (long long)blockIdx.y * tps * TILE;\n"
    << "  const long long jend = n < jbeg + tps * TILE ? n : jbeg + tps * TILE;\n"
    << "  for (long long j0 = jbeg; j0 < jend; j0 += TILE) {\n"
    << "    __syncthreads();\n"
    << "    for (int q = threadIdx.x; q < TILE * DP; q += blockDim.x) {\n"
    << "      const int jj = q / DP, k = q - jj * DP;\n"
    << "      const long long j = j0 + jj;\n"
    << "      sx[q] = (j < n && k < D) ? Xc[j * D + k] : 0.0f;\n"
    << "    }\n"
    << "    for (int q = threadIdx.x; q < TILE * NC; q += blockDim.x) {\n"
    << "      const int c = q / TILE, jj = q - c * TILE;\n"
    << "      const long long j = j0 + jj;\n"
    << "      sv[q] = (c < nc && j < n) ? V[(long long)c * n + j] : 0.0f;\n"
    << "    }\n"
    << "    __syncthreads();\n"
    << "    float pa[NC];\n"
    << "#pragma unroll\n"
    << "    for (int c = 0; c < NC; ++c) pa[c] = 0.0f;\n"
    << "    const int cnt = (int)(jend - j0 < TILE ? jend - j0 : TILE);\n"
    << "#pragma unroll 2\n"
    << "    for (int jj = 0; jj < cnt; ++jj) {\n"
    << "      const float k = kval(xi, sx + jj * DP);\n"
    << "#pragma unroll\n"
    << "      for (int c = 0; c < NC; ++c) pa[c] = fmaf(k, sv[c * TILE + jj], pa[c]);\n"
    << "    }\n"
    << "#pragma unroll\n"
    << "    for (int c = 0; c < NC; ++c) acc[c] += (double)pa[c];\n"
    << "  }\n"
    << "  if (i < m) {\n"
    << "    float* dst = part + (long long)blockIdx.y * nc * m;\n"
    << "#pragma unroll\n"
    << "    for (int c = 0; c < NC; ++c)\n"
    << "      if (c < nc) dst[(long long)c * m + i] = (float)acc[c];\n"
    << "  }\n"
    << "}\n";
  // 8..16 right-hand sides: the product on the fp32 matrix cores.  Wave w
  // owns row tiles i0 + 16 r (r < R); per step of 4 columns j = j0 + 4 s +
  // l/16 each lane evaluates the pair (row i0 + 16 r + l%16, column j) as the
  // A operand of v_mfma_f32_16x16x4_f32 and supplies B = V[l%16][j]; D holds
  // rows i0 + 16 r + 4 (l/16) + q of right-hand side l%16.  Per column tile
  // the fp32 D is added into fp64.
  s << "typedef float f4m __attribute__((ext_vector_type(4)));\n"
    << "#define R " << kJitMfmaRowTiles << "\n"
    << "__device__ __forceinline__ void body_mfma(const float* __restrict__ Xr, long long m,\n"
    << "    const float* __restrict__ Xc, long long n, const float* __restrict__ p,\n"
    << "    const float* __restrict__ V, int nc, float* __restrict__ part) {\n"
    << "  extern __shared__ float sm[];\n"
    << "  float* sx = sm;\n"
    << "  float* sv = sm + TILE * DP;\n"
    << pro
    << "  auto kval = [&](const float* __restrict__ xi, const float* __restrict__ xj)\n"
    << "      __attribute__((always_inline)) -> float {\n"
    << pair
    << "  };\n"
    << "  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;\n"
    << "  const int lm = lane & 15, lq = lane >> 4;\n"
    << "  const long long i0 = ((long long)blockIdx.x * 4 + wave) * (16 * R);\n"
    << "  float xi[R][DP];\n"
    << "#pragma unroll\n"
    << "  for (int r = 0; r < R; ++r) {\n"
    << "    const long long i = i0 + 16 * r + lm;\n"
    << "#pragma unroll\n"
    << "    for (int k = 0; k < DP; ++k) xi[r][k] = (i < m && k < D) ? Xr[i * D + k] : 0.0f;\n"
    << "  }\n"
    << "  double acc[R][4];\n"
    << "#pragma unroll\n"
    << "  for (int r = 0; r < R; ++r)\n"
    << "#pragma unroll\n"
    << "    for (int q = 0; q < 4; ++q) acc[r][q] = 0.0;\n"
    << "  const long long tiles = (n + TILE - 1) / TILE;\n"
    << "  const long long tps = (tiles + gridDim.y - 1) / gridDim.y;\n"
    << "  const long long jbeg = (long long)blockIdx.y * tps * TILE;\n"
    << "  const long long jend = n < jbeg + tps * TILE ? n : jbeg + tps * TILE;\n"
    << "  for (long long j0 = jbeg; j0 < jend; j0 += TILE) {\n"
    << "    __syncthreads();\n"
    << "    for (int q = threadIdx.x; q < TILE * DP; q += blockDim.x) {\n"
    << "      const int jj = q / DP, k = q - jj * DP;\n"
    << "      const long long j = j0 + jj;\n"
    << "      sx[q] = (j < n && k < D) ? Xc[j * D + k] : 0.0f;\n"
    << "    }\n"
    << "    for (int q = threadIdx.x; q < TILE * 16; q += blockDim.x) {\n"
    << "      const int c = q / TILE, jj = q - c * TILE;\n"
    << "      const long long j = j0 + jj;\n"
    << "      sv[q] = (c < nc && j < jend) ? V[(long long)c * n + j] : 0.0f;\n"
    << "    }\n"
    << "    __syncthreads();\n"
    << "    f4m d[R];\n"
    << "#pragma unroll\n"
    << "    for (int r = 0; r < R; ++r) d[r] = f4m{0.0f, 0.0f, 0.0f, 0.0f};\n"
    << "    const int steps = (int)((jend - j0 < TILE ? jend - j0 : TILE) + 3) / 4;\n"
    << "#pragma unroll 2\n"
    << "    for (int st = 0; st < steps; ++st) {\n"
    << "      const int jj = 4 * st + lq;\n"
    << "      const float* xj = sx + jj * DP;\n"
    << "      const float b = sv[lm * TILE + jj];\n"
    << "#pragma unroll\n"
    << "      for (int r = 0; r < R; ++r)\n"
    << "        d[r] = __builtin_amdgcn_mfma_f32_16x16x4f32(kval(xi[r], xj), b, d[r], 0, 0, 0);\n"
    << "    }\n"
    << "#pragma unroll\n"
    << "    for (int r = 0; r < R; ++r)\n"
    << "#pragma unroll\n"
    << "      for (int q = 0; q < 4; ++q) acc[r][q] += (double)d[r][q];\n"
    << "  }\n"
    << "  if (lm < nc) {\n"
    << "    float* dst = part + ((long long)blockIdx.y * nc + lm) * m;\n"
    << "#pragma unroll\n"
    << "    for (int r = 0; r < R; ++r)\n"
    << "#pragma unroll\n"
    << "      for (int q = 0; q < 4; ++q) {\n"
    << "        const long long i = i0 + 16 * r + 4 * lq + q;\n"
    << "        if (i < m) dst[i] = (float)acc[r][q];\n"
    << "      }\n"
    << "  }\n"
    << "}\n";
  for (int nc : kJitCols) {
    s << "extern \"C\" __global__ __launch_bounds__(256) void k_tree_jit_" << nc
      << "(const float* Xr, long long m, const float* Xc, long long n, const float* p,\n"
      << "    const float* V, int nc, float* part) { ";
    if (nc >= kJitMfmaMinCols)
      s << "body_mfma(Xr, m, Xc, n, p, V, nc, part); }\n";
    else
      s << "body<" << nc << ">(Xr, m, Xc, n, p, V, nc, part); }\n";
  }
  return s.str();
}

// Backward pass of one pair and the final factors of its sums: the pair code
// (after emit_tree's) adds w dK/dtheta_q, less a factor that depends on the
// parameters only, into g[q]; fin holds that factor per parameter (C
// expressions of p in double: rounded to fp32 it would scale the whole sum by
// up to 1 + 2^-24), applied once per thread.  False when two leaves or
// scales share a parameter slot (their factors differ).
bool emit_tree_grad(const KernelTree& t, std::string& pair, std::vector<std::string>& fin) {
  std::ostringstream Q;
  fin.assign((size_t)t.nparams, "0.0f");
  std::vector<char> used((size_t)t.nparams, 0);
  bool ok = true;
  auto own = [&](int q, const std::string& factor) {
    if (q < 0 || q >= t.nparams || used[(size_t)q]) {
      ok = false;
      return;
    }
    used[(size_t)q] = 1;
    fin[(size_t)q] = factor;
  };
  auto pq = [](int q) { return "(double)p[" + std::to_string(q) + "]"; };
  for (int i = 0; i < t.nnodes; ++i)
    Q << "  float a" << i << " = " << (i == t.nnodes - 1 ? "w" : "0.0f") << ";\n";
  for (int i = t.nnodes - 1; i >= 0; --i) {
    const TreeNode& nd = t.node[i];
    const std::string A = "a" + std::to_string(i);
    if (nd.code == TN_ADD) {
      Q << "  a" << nd.a << " += " << A << "; a" << nd.b << " += " << A << ";\n";
      continue;
    }
    if (nd.code == TN_MUL) {
      Q << "  a" << nd.a << " = fmaf(" << A << ", n" << nd.b << ", a" << nd.a << "); a" << nd.b
        << " = fmaf(" << A << ", n" << nd.a << ", a" << nd.b << ");\n";
      continue;
    }
    if (nd.code == TN_SCALE) {
      Q << "  a" << nd.a << " = fmaf(" << A << ", s" << i << ", a" << nd.a << ");\n  g[" << nd.b
        << "] = fmaf(" << A << ", n" << nd.a << ", g[" << nd.b << "]);\n";
      own(nd.b, "1.0f");
      continue;
    }
    const int l = nd.a;
    const TreeLeaf& lf = t.leaf[l];
    if (lf.kind == KIND_CAT) continue;  // tables are learned outside this pass
    const std::string L = "l" + std::to_string(l);
    const int nls = lf.ard ? lf.ndim : 1;
    auto add = [&](int q, const std::string& x, const std::string& y, const std::string& factor) {
      Q << "  g[" << q << "] = fmaf(" << x << ", " << y << ", g[" << q << "]);\n";
      own(q, factor);
    };
    if (lf.kind == KIND_LINEAR || lf.kind == KIND_POLY) {
      const bool poly = lf.kind == KIND_POLY;
      const int ios = lf.p0 + nls + (poly ? 2 : 0);
      std::string h = A, factor = pq(ios);
      if (poly) {
        Q << "  const float " << L << "h = " << A << " * " << L << "bp;\n";
        h = L + "h";
        factor = f((float)lf.deg) + " * " + pq(ios);
        Q << "  g[" << lf.p0 + nls + 1 << "] += " << h << ";\n";
        own(lf.p0 + nls + 1, factor);
      }
      for (int q = 0; q < nls; ++q)
        add(lf.p0 + q, h, lf.ard ? L + "x" + std::to_string(q) : L + "raw", factor);
      add(ios, A, L, "1.0 / " + pq(ios));
      continue;
    }
    if (lf.kind == KIND_PERIODIC) {
      const int ip = lf.p0 + nls, ios = ip + 1;
      // k = os exp(-2 S), S = sum_q sin^2(t_q) / l_q, t_q = pi dx_q / period
      Q << "  const float " << L << "h = " << A << " * " << L << ";\n  float " << L
        << "c = 0.0f;\n";
      for (int q = 0; q < lf.ndim; ++q) {
        const std::string n = L + "n" + std::to_string(q), tq = L + "t" + std::to_string(q);
        Q << "  " << L << "c = fmaf(" << n << " * __cosf(" << tq << "), " << tq << " * " << L
          << "il" << (lf.ard ? q : 0) << ", " << L << "c);\n";
        if (lf.ard)
          add(lf.p0 + q, L + "h * " + n, n,
              "2.0 / (" + pq(lf.p0 + q) + " * " + pq(lf.p0 + q) + ")");
      }
      if (!lf.ard) add(lf.p0, L + "h", L + "s", "2.0 / " + pq(lf.p0));
      add(ip, L + "h", L + "c", "4.0 / " + pq(ip));
      Q << "  g[" << ios << "] += " << L << "h;\n";
      own(ios, "1.0 / " + pq(ios));
      continue;
    }
    // radial / RQ lengthscales: dk/dl_q = h u_q^2 / l_q with u_q = dx_q / l_q
    int ios = lf.p0 + nls;
    Q << "  const float " << L << "a = " << A << " * " << L << ";\n  const float " << L << "h = ";
    if (lf.kind == KIND_RBF) {
      Q << L << "a;\n";
    } else if (lf.kind == KIND_MATERN12) {
      Q << L << "a * __builtin_amdgcn_rcpf(" << L << "r);\n";
    } else if (lf.kind == KIND_MATERN32) {
      Q << A << " * (3.0f * " << L << "os) * " << L << "e;\n";
    } else if (lf.kind == KIND_RQ) {
      ios += 1;
      Q << L << "a * __builtin_amdgcn_rcpf(" << L << "B);\n";
      // dk/dalpha = k (r^2 / (2 alpha B) - ln B)
      add(lf.p0 + nls, L + "a",
          "fmaf(" + L + "r2 * " + L + "ia, __builtin_amdgcn_rcpf(" + L + "B), " + f(-kLn2) +
              " * " + L + "lb)",
          "1.0f");
    } else {
      Q << A << " * (5.0f / 3.0f * " << L << "os) * (1.0f + " << L << "s5) * " << L << "e;\n";
    }
    if (lf.ard)
      for (int q = 0; q < lf.ndim; ++q) {
        const std::string u = L + "u" + std::to_string(q);
        add(lf.p0 + q, L + "h * " + u, u, "1.0 / " + pq(lf.p0 + q));
      }
    else
      add(lf.p0, L + "h", L + "r2", "1.0 / " + pq(lf.p0));
    Q << "  g[" << ios << "] += " << L << "a;\n";
    own(ios, "1.0 / " + pq(ios));
  }
  pair = Q.str();
  return ok;
}

// Gradient-trace kernel of the tree: part[(y gx + x) P + q] = the block's
// share of sum_ab dK_ab/dtheta_q sum_c Lf[c][a] Rf[c][b], c in [c0, ncols).
//
// Every evaluator of a pair costs the forward and backward pass of the tree
// (~100 VALU instructions for two or three leaves), so the kernel is VALU
// bound and a pair is formed once for both of its orders where the tree is
// symmetric (no correlation tables; n = 10007, RBF x periodic + RQ, 11 factor
// columns: 7.54 ms interpreted, 0.22 ms): blocks of 128 points, row block b taking
// the column blocks (b + delta) mod nb of the cyclic half, its diagonal block
// with weight 1/2.  Per 16 x 16 tile w_ab + w_ba comes from the fp32 matrix
// cores (v_mfma_f32_16x16x4_f32 over the factor columns, four at a time), its
// result w[q] belonging to the pair (column 4 (lane/16) + q, row lane%16), so
// a lane keeps its rows in registers and reads columns from LDS.  g sums a
// lane's 8 pairs of a tile column in fp32, then fp64.
std::string tree_grad_source(const KernelTree& t) {
  std::string pro, pair, back;
  std::vector<std::string> fin;
  emit_tree(t, pro, pair);
  if (!emit_tree_grad(t, back, fin)) return std::string();
  const int D = t.d, DP = (D + 3) / 4 * 4, P = t.nparams;
  const bool sym = t.table_size == 0;
  std::ostringstream s;
  s << "#define D " << D << "\n#define DP " << DP << "\n#define P " << P << "\n#define BLK "
    << kTreeGradBlock << "\n#define SYM " << (sym ? 1 : 0) << "\n"
    << R"(typedef float f4m __attribute__((ext_vector_type(4)));
#define R 2
#define CS (BLK + 16)
extern "C" __global__ __launch_bounds__(256) void k_tree_grad_jit(
    const float* __restrict__ X, long long n, const float* __restrict__ p,
    const float* __restrict__ Lf, const float* __restrict__ Rf, int ncols, int c0, long long nb,
    long long dps, double* __restrict__ part) {
  __shared__ __align__(16) float sx[BLK * DP];
  __shared__ float sl[16 * CS], sr[16 * CS];
  __shared__ double red[4];
)" << pro
    << R"(  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int lm = lane & 15, lq = lane >> 4;
  const int cn = ncols - c0 < 16 ? ncols - c0 : 16;
  const int csteps = (cn + 3) / 4;
  const long long b = blockIdx.x;
  float xi[R][DP], lb[R][4], rb[R][4];
#pragma unroll
  for (int r = 0; r < R; ++r) {
    const long long i = b * BLK + (wave * R + r) * 16 + lm;
#pragma unroll
    for (int k = 0; k < DP; ++k) xi[r][k] = (i < n && k < D) ? X[i * D + k] : 0.0f;
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      const int c = 4 * s + lq;
      const bool in = i < n && c < cn;
      lb[r][s] = in ? Lf[(long long)(c0 + c) * n + i] : 0.0f;
      rb[r][s] = in ? Rf[(long long)(c0 + c) * n + i] : 0.0f;
    }
  }
  double gd[P];
#pragma unroll
  for (int q = 0; q < P; ++q) gd[q] = 0.0;
#if SYM
  const long long span = (nb & 1) ? (nb - 1) / 2 : (b < nb / 2 ? nb / 2 : nb / 2 - 1);
#else
  const long long span = nb - 1;
#endif
  const long long d0 = (long long)blockIdx.y * dps;
  const long long d1 = d0 + dps < span + 1 ? d0 + dps : span + 1;
  for (long long dl = d0; dl < d1; ++dl) {
    long long J = b + dl;
    if (J >= nb) J -= nb;
    const long long j0 = J * BLK;
    const int cnt = (int)(n - j0 < BLK ? n - j0 : BLK);
    __syncthreads();
    for (int q = threadIdx.x; q < BLK * DP; q += 256) {
      const int jj = q / DP, k = q - jj * DP;
      sx[q] = (jj < cnt && k < D) ? X[(j0 + jj) * D + k] : 0.0f;
    }
    for (int q = threadIdx.x; q < BLK * 16; q += 256) {
      const int c = q / BLK, jj = q - c * BLK;
      const bool in = jj < cnt && c < cn;
      sr[c * CS + jj] = in ? Rf[(long long)(c0 + c) * n + j0 + jj] : 0.0f;
#if SYM
      sl[c * CS + jj] = in ? Lf[(long long)(c0 + c) * n + j0 + jj] : 0.0f;
#endif
    }
    __syncthreads();
    const float wt = (SYM && dl == 0) ? 0.5f : 1.0f;
    const int tiles = (cnt + 15) / 16;
#pragma unroll 1
    for (int ct = 0; ct < tiles; ++ct) {
      float g[P];
#pragma unroll
      for (int q = 0; q < P; ++q) g[q] = 0.0f;
      f4m wv[R];
#pragma unroll
      for (int r = 0; r < R; ++r) wv[r] = f4m{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
      for (int s = 0; s < 4; ++s) {
        if (s >= csteps) break;
        const float ar = sr[(4 * s + lq) * CS + 16 * ct + lm];
#if SYM
        const float al = sl[(4 * s + lq) * CS + 16 * ct + lm];
#endif
#pragma unroll
        for (int r = 0; r < R; ++r) {
          wv[r] = __builtin_amdgcn_mfma_f32_16x16x4f32(ar, lb[r][s], wv[r], 0, 0, 0);
#if SYM
          wv[r] = __builtin_amdgcn_mfma_f32_16x16x4f32(al, rb[r][s], wv[r], 0, 0, 0);
#endif
        }
      }
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const float* xjp = sx + (16 * ct + 4 * lq + e) * DP;
        float xj[DP];
#pragma unroll
        for (int k = 0; k < DP; k += 4) {
          const f4m x = *reinterpret_cast<const f4m*>(xjp + k);
          xj[k] = x[0]; xj[k + 1] = x[1]; xj[k + 2] = x[2]; xj[k + 3] = x[3];
        }
#pragma unroll
        for (int r = 0; r < R; ++r) {
          const float w = wt * wv[r][e];
          auto one = [&](const float* xi) __attribute__((always_inline)) {
)" << pair << back
    << R"(          };
          one(xi[r]);
        }
      }
#pragma unroll
      for (int q = 0; q < P; ++q) gd[q] += (double)g[q];
    }
  }
  double* dst = part + ((long long)blockIdx.y * gridDim.x + blockIdx.x) * P;
  auto put = [&](int q, double v) {
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) v += __shfl_xor(v, o);
    __syncthreads();
    if (lane == 0) red[wave] = v;
    __syncthreads();
    if (threadIdx.x == 0) dst[q] = red[0] + red[1] + red[2] + red[3];
  };
)";
  for (int q = 0; q < P; ++q)
    s << "  put(" << q << ", gd[" << q << "] * (double)(" << fin[(size_t)q] << "));\n";
  s << "}\n";
  return s.str();
}

// Symmetric product kernel of the tree (square products, stationary in the
// sense K_ij = K_ji): every off-diagonal value is formed once and used for both
// of its entries.  A value costs ~15 VALU instructions per leaf and dimension
// beside the 64 cycles a pair of fp32 matrix instructions spends on it, so
// halving the values is worth the transposition.  Blocks of 256 points, row
// block b taking stages [g0, g1) (64 columns each) of its own block and of the
// column blocks (b + delta) mod nb of the cyclic half.  Per 16 x 16 tile a lane
// evaluates the pairs (row lane%16, columns 4 (lane/16) + s), the A operands of
// out_I += K V_J; their rows go through a wave-private LDS tile (stride 20:
// conflict-free both ways) and come back as the A operands of out_J += K^T V_I
// with the rows' right-hand sides in registers.  The waves' transposed sums
// are added in LDS and written per stage: tp[((b hmax + delta - 1) 256 + j) 16
// + c]; forward sums (fp64 across stages) fwd[(split 16 + c) npad + i].
std::string tree_sym_source(const KernelTree& t) {
  std::string pro, pair;
  emit_tree(t, pro, pair);
  pair += tree_value_return(t);
  const int D = t.d, DP = (D + 3) / 4 * 4;
  std::ostringstream s;
  s << "#define D " << D << "\n#define DP " << DP << "\n#define BLK " << kTreeSymBlock
    << "\n#define R " << kTreeSymBlock / 64 << "\n#define ST " << kTreeSymStage << "\n"
    << R"(typedef float f4m __attribute__((ext_vector_type(4)));
#define VS 20
// a wave's LDS stores before its later loads of other lanes' words
__device__ __forceinline__ void wave_lds_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}
extern "C" __global__ __launch_bounds__(256) void k_tree_sym_jit(
    const float* __restrict__ X, long long n, const float* __restrict__ p,
    const float* __restrict__ V, int nc, long long nb, long long splits, long long sps,
    long long hmax, float* __restrict__ fwd, float* __restrict__ tp) {
  __shared__ __align__(16) float sx[ST * DP];
  __shared__ __align__(16) float sv[ST * VS];
  __shared__ __align__(16) float tsc[4][2][16 * VS];
  __shared__ __align__(16) f4m tbuf[4][ST / 16][64];
)" << pro
    << R"(  auto kval = [&](const float* __restrict__ xi, const float* __restrict__ xj)
      __attribute__((always_inline)) -> float {
)" << pair
    << R"(  };
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int lm = lane & 15, lq = lane >> 4;
  const long long b = blockIdx.x, split = blockIdx.y, npad = nb * BLK;
  const long long i0 = b * BLK + wave * (16 * R);
  float xi[R][DP], vr[R][4];
#pragma unroll
  for (int r = 0; r < R; ++r) {
    const long long i = i0 + 16 * r + lm;
#pragma unroll
    for (int k = 0; k < DP; ++k) xi[r][k] = (i < n && k < D) ? X[i * D + k] : 0.0f;
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      const long long ii = i0 + 16 * r + 4 * lq + s;
      vr[r][s] = (ii < n && lm < nc) ? V[(long long)lm * n + ii] : 0.0f;
    }
  }
  double acc[R][4];
#pragma unroll
  for (int r = 0; r < R; ++r)
#pragma unroll
    for (int q = 0; q < 4; ++q) acc[r][q] = 0.0;
  const int per = BLK / ST;
  const long long span = (nb & 1) ? (nb - 1) / 2 : (b < nb / 2 ? nb / 2 : nb / 2 - 1);
  const long long g0 = split * sps, gl = (span + 1) * per;
  const long long g1 = g0 + sps < gl ? g0 + sps : gl;
  for (long long g = g0; g < g1; ++g) {
    const long long dl = g / per;
    long long J = b + dl;
    if (J >= nb) J -= nb;
    const long long j0 = J * BLK + (g % per) * ST;
    // (the previous stage's operands are free: its second barrier)
    for (int q = threadIdx.x; q < ST * DP; q += 256) {
      const int jj = q / DP, k = q - jj * DP;
      sx[q] = (j0 + jj < n && k < D) ? X[(j0 + jj) * D + k] : 0.0f;
    }
    for (int q = threadIdx.x; q < ST * 16; q += 256) {
      const int c = q / ST, jj = q - c * ST;
      sv[jj * VS + c] = (c < nc && j0 + jj < n) ? V[(long long)c * n + j0 + jj] : 0.0f;
    }
    __syncthreads();
    f4m d1[R];
#pragma unroll
    for (int r = 0; r < R; ++r) d1[r] = f4m{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll 1
    for (int ct = 0; ct < ST / 16; ++ct) {
      f4m d2 = f4m{0.0f, 0.0f, 0.0f, 0.0f};
      float kv[R][4];
#pragma unroll
      for (int s = 0; s < 4; ++s) {
        const int jj = 16 * ct + 4 * lq + s;
        float xj[DP];
#pragma unroll
        for (int k = 0; k < DP; k += 4) {
          const f4m x = *reinterpret_cast<const f4m*>(sx + jj * DP + k);
          xj[k] = x[0]; xj[k + 1] = x[1]; xj[k + 2] = x[2]; xj[k + 3] = x[3];
        }
        const float v = sv[jj * VS + lm];
#pragma unroll
        for (int r = 0; r < R; ++r) {
          kv[r][s] = kval(xi[r], xj);
          d1[r] = __builtin_amdgcn_mfma_f32_16x16x4f32(kv[r][s], v, d1[r], 0, 0, 0);
        }
      }
      if (dl > 0) {
#pragma unroll
        for (int r = 0; r < R; ++r) {
          float* sc = tsc[wave][r & 1];
          *reinterpret_cast<f4m*>(sc + lm * VS + 4 * lq) =
              f4m{kv[r][0], kv[r][1], kv[r][2], kv[r][3]};
          wave_lds_sync();  // (the other buffer's reads, too, stay before its next store)
#pragma unroll
          for (int s = 0; s < 4; ++s)
            d2 = __builtin_amdgcn_mfma_f32_16x16x4f32(sc[(4 * lq + s) * VS + lm], vr[r][s], d2, 0,
                                                      0, 0);
        }
        tbuf[wave][ct][lane] = d2;
      }
    }
#pragma unroll
    for (int r = 0; r < R; ++r)
#pragma unroll
      for (int q = 0; q < 4; ++q) acc[r][q] += (double)d1[r][q];
    __syncthreads();
    if (dl > 0) {
      // lane of column tile ct: columns 4 (lane/16) + q, right-hand side lane%16
      float* dst = tp + ((b * hmax + dl - 1) * BLK + (g % per) * ST) * 16;
      for (int q = threadIdx.x; q < ST * 4; q += 256) {
        const int ct = q >> 6, ln = q & 63;
        const f4m a = tbuf[0][ct][ln], bb = tbuf[1][ct][ln], c = tbuf[2][ct][ln],
                  e = tbuf[3][ct][ln];
#pragma unroll
        for (int k = 0; k < 4; ++k)
          dst[(16 * ct + 4 * (ln >> 4) + k) * 16 + (ln & 15)] =
              (float)((double)a[k] + (double)bb[k] + (double)c[k] + (double)e[k]);
      }
    }
  }
#pragma unroll
  for (int r = 0; r < R; ++r)
#pragma unroll
    for (int q = 0; q < 4; ++q)
      fwd[(split * 16 + lm) * npad + i0 + 16 * r + 4 * lq + q] = (float)acc[r][q];
}
)";
  return s.str();
}

std::string spec_key(const KernelTree& t) {
  std::ostringstream o;
  o << t.d << ' ' << t.nparams << ' ' << t.nleaves << ' ' << t.nnodes << ' ' << t.table_size;
  for (int l = 0; l < t.nleaves; ++l) {
    const TreeLeaf& lf = t.leaf[l];
    o << " L" << lf.kind << ',' << lf.ard << ',' << lf.ndim << ',' << lf.dim_off << ','
      << lf.p0 << ',' << lf.deg;
  }
  for (int i = 0; i < t.nnodes; ++i) o << " N" << t.node[i].code << ',' << t.node[i].a << ','
                                       << t.node[i].b;
  int nd = 0;
  for (int l = 0; l < t.nleaves; ++l) nd += t.leaf[l].ndim;
  for (int q = 0; q < nd; ++q) o << " d" << t.dims[q];
  return o.str();
}

struct Compiled {
  hipModule_t mod = nullptr;
  hipFunction_t fn[5] = {};
};

std::mutex g_jit_mu;
std::map<std::pair<std::string, int>, Compiled> g_jit;

#define MGP_RTC_CHECK(expr, prog)                                                         \
  do {                                                                                    \
    const hiprtcResult r_ = (expr);                                                       \
    if (r_ != HIPRTC_SUCCESS) {                                                           \
      std::string log_;                                                                   \
      size_t n_ = 0;                                                                      \
      if (prog && hiprtcGetProgramLogSize(prog, &n_) == HIPRTC_SUCCESS && n_ > 1) {        \
        log_.resize(n_);                                                                  \
        (void)hiprtcGetProgramLog(prog, &log_[0]);                                        \
      }                                                                                   \
      throw Error(ST_INTERNAL, std::string("hiprtc: ") + hiprtcGetErrorString(r_) + " in " \
                                   #expr + (log_.empty() ? "" : "\n" + log_));            \
    }                                                                                     \
  } while (0)

hipModule_t compile_source(const std::string& src, const char* name) {
  hiprtcProgram prog = nullptr;
  MGP_RTC_CHECK(hiprtcCreateProgram(&prog, src.c_str(), name, 0, nullptr, nullptr), prog);
  // packed-FP32 VALU forms are disabled here as for every device file
  const char* opts[] = {"--offload-arch=gfx950", "-O3", "-std=c++17", "-Xclang",
                        "-target-feature", "-Xclang", "-packed-fp32-ops"};
  const hiprtcResult rc = hiprtcCompileProgram(prog, (int)(sizeof(opts) / sizeof(opts[0])), opts);
  std::vector<char> code;
  try {
    MGP_RTC_CHECK(rc, prog);
    size_t size = 0;
    MGP_RTC_CHECK(hiprtcGetCodeSize(prog, &size), prog);
    code.resize(size);
    MGP_RTC_CHECK(hiprtcGetCode(prog, code.data()), prog);
  } catch (...) {
    (void)hiprtcDestroyProgram(&prog);
    throw;
  }
  (void)hiprtcDestroyProgram(&prog);
  hipModule_t mod = nullptr;
  MGP_HIP_CHECK(hipModuleLoadData(&mod, code.data()));
  return mod;
}

Compiled compile_tree(const KernelTree& t) {
  Compiled c;
  c.mod = compile_source(tree_source(t), "kernel_tree_jit.hip");
  for (int k = 0; k < 5; ++k) {
    const std::string name = "k_tree_jit_" + std::to_string(kJitCols[k]);
    MGP_HIP_CHECK(hipModuleGetFunction(&c.fn[k], c.mod, name.c_str()));
  }
  return c;
}

// Gradient kernels per (tree, device); fn null where the tree has none.
std::map<std::pair<std::string, int>, hipFunction_t> g_jit_grad;
// Symmetric product kernels and their workgroups per CU.
std::map<std::pair<std::string, int>, std::pair<hipFunction_t, int>> g_jit_sym;

}  // namespace

std::string tree_jit_source(const KernelTree& t) { return tree_source(t); }
std::string tree_grad_jit_source(const KernelTree& t) { return tree_grad_source(t); }
std::string tree_sym_jit_source(const KernelTree& t) { return tree_sym_source(t); }

TreeSymJitKernel tree_sym_jit_kernel(const KernelTree& t) {
  MGP_REQUIRE(t.table_size == 0, "correlation tables need not be symmetric");
  int dev = 0;
  MGP_HIP_CHECK(hipGetDevice(&dev));
  const auto key = std::make_pair(spec_key(t), dev);
  std::lock_guard<std::mutex> lk(g_jit_mu);
  auto it = g_jit_sym.find(key);
  if (it == g_jit_sym.end()) {
    hipFunction_t fn = nullptr;
    MGP_HIP_CHECK(hipModuleGetFunction(
        &fn, compile_source(tree_sym_source(t), "kernel_tree_sym_jit.hip"), "k_tree_sym_jit"));
    int per_cu = 0;
    MGP_HIP_CHECK(hipModuleOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, fn, 256, 0));
    it = g_jit_sym.emplace(key, std::make_pair(fn, std::max(per_cu, 1))).first;
  }
  TreeSymJitKernel out;
  out.fn = it->second.first;
  out.per_cu = it->second.second;
  out.block = kTreeSymBlock;
  out.stage = kTreeSymStage;
  return out;
}

TreeGradJitKernel tree_grad_jit_kernel(const KernelTree& t) {
  int dev = 0;
  MGP_HIP_CHECK(hipGetDevice(&dev));
  const auto key = std::make_pair(spec_key(t), dev);
  std::lock_guard<std::mutex> lk(g_jit_mu);
  auto it = g_jit_grad.find(key);
  if (it == g_jit_grad.end()) {
    hipFunction_t fn = nullptr;
    const std::string src = tree_grad_source(t);
    if (!src.empty())
      MGP_HIP_CHECK(hipModuleGetFunction(&fn, compile_source(src, "kernel_tree_grad_jit.hip"),
                                         "k_tree_grad_jit"));
    it = g_jit_grad.emplace(key, fn).first;
  }
  TreeGradJitKernel out;
  out.fn = it->second;
  out.block = kTreeGradBlock;
  out.symmetric = t.table_size == 0;
  return out;
}

TreeJitKernel tree_jit_kernel(const KernelTree& t, int nc) {
  MGP_REQUIRE(nc >= 1 && nc <= 16, "tree product pass takes 1..16 right-hand sides");
  int dev = 0;
  MGP_HIP_CHECK(hipGetDevice(&dev));
  const auto key = std::make_pair(spec_key(t), dev);
  std::lock_guard<std::mutex> lk(g_jit_mu);
  auto it = g_jit.find(key);
  if (it == g_jit.end()) it = g_jit.emplace(key, compile_tree(t)).first;
  int k = 0;
  while (kJitCols[k] < nc) ++k;
  TreeJitKernel out;
  out.fn = it->second.fn[k];
  out.ncols = kJitCols[k];
  const int DP = (t.d + 3) / 4 * 4;
  const bool mfma = out.ncols >= kJitMfmaMinCols;
  out.rows_per_block = mfma ? 4 * 16 * kJitMfmaRowTiles : 256;
  out.lds_bytes = (size_t)kJitTile * (DP + (mfma ? 16 : out.ncols)) * sizeof(float);
  return out;
}

}  // namespace mgp
