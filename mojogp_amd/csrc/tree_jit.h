// Run-time compiled (hiprtc) product kernels of composite kernel trees.
#pragma once

#include <string>

#include "kernel_tree.h"

namespace mgp {

struct TreeJitKernel {
  hipFunction_t fn = nullptr;  // extern "C" k_tree_jit_<ncols>
  int ncols = 0;               // right-hand sides the kernel accumulates (>= requested)
  size_t lds_bytes = 0;        // dynamic LDS per 256-thread block
  int rows_per_block = 256;    // rows of Xr per block (grid x = ceil(m / rows_per_block))
};

// The straight-line product kernel of tree t for nc <= 16 right-hand sides:
// arguments (const float* Xr, long long m, const float* Xc, long long n,
// const float* p, const float* V, int nc, float* part), grid
// (ceil(m / rows_per_block), column splits), 256 threads; part[y][c][i] = split y's sum over its columns
// j of K(Xr_i, Xc_j) V[c][j].  Compiled on first use per (tree, device).
TreeJitKernel tree_jit_kernel(const KernelTree& t, int nc);
// The generated source (tests and inspection).
std::string tree_jit_source(const KernelTree& t);

struct TreeSymJitKernel {
  hipFunction_t fn = nullptr;  // extern "C" k_tree_sym_jit
  int per_cu = 1;              // workgroups a CU holds
  int block = 0, stage = 0;    // points per block, columns per stage
};

// The symmetric product kernel of tree t (no correlation tables) for up to 16
// right-hand sides: arguments (const float* X, long long n, const float* p,
// const float* V, int nc, long long nb, long long splits, long long sps, long
// long hmax, float* fwd, float* tp), grid (nb, splits), 256 threads; see
// tree_sym_source for the layouts.  Compiled on first use per (tree, device).
TreeSymJitKernel tree_sym_jit_kernel(const KernelTree& t);
std::string tree_sym_jit_source(const KernelTree& t);

struct TreeGradJitKernel {
  hipFunction_t fn = nullptr;  // extern "C" k_tree_grad_jit; null: not generated for this tree
  int block = 0;               // points per block
  bool symmetric = false;      // column blocks of the cyclic half only
};

// The straight-line gradient-trace kernel of tree t: arguments (const float*
// X, long long n, const float* p, const float* Lf, const float* Rf, int
// ncols, int c0, long long nb, long long dps, double* part), grid (nb =
// ceil(n / block), splits of dps column-block offsets), 256 threads;
// part[(y nb + x) P + q] = the block's share of parameter q's trace over the
// factor columns c0 .. min(c0 + 16, ncols).  Compiled on first use per (tree,
// device); null for trees whose leaves share parameter slots.
TreeGradJitKernel tree_grad_jit_kernel(const KernelTree& t);
std::string tree_grad_jit_source(const KernelTree& t);

}  // namespace mgp
