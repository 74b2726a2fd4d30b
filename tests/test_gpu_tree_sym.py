"""Symmetric generated products of kernel trees (square, 5 .. 16 right-hand
sides, from 5800 to 6500 points on for these trees) at the edges of their
256-point blocks and 64-column stages (even and odd block counts, ragged last
block), beside column chunks and sizes that stay on the one-sided kernel,
against the float64 tree restatement on sampled rows;
a tree with a correlation table keeps the one-sided kernel.

Bound: a value carries the hardware exp / sin / log error and an exponent
within a few units, ~16 ulps = 1e-6; the sums average it."""

import numpy as np
import pytest

from mojogp_amd import GD, RBF, RQ, Linear, Matern12, Matern52, Periodic, Polynomial, make_ard_kernel
from mojogp_amd import _lib
from mojogp_amd._provider import NativeProvider
from oracle import kernels as ok

pytestmark = pytest.mark.gpu

TREES = {
    "rbf*per[0]+rq": (lambda: RBF() * Periodic(active_dims=[0]) + RQ(), 3),
    "ard 9-d": (lambda: make_ard_kernel(RBF(ard=True) + 2.0 * Matern52(ard=True), 9), 9),
    "m12*poly+lin": (lambda: Matern12() * Polynomial(degree=2.0) + Linear(), 2),
}


def _run(node, T, d, X, V, params, tables=None):
    n = len(X)
    p = NativeProvider(None, False, X, params, 0.3, tree_spec=node.to_tree_spec(d))
    try:
        if tables is not None:
            flat = np.ascontiguousarray(tables.ravel())
            _lib.call("mgp_set_categorical_tables", p.handle, _lib.fptr(flat), int(flat.size))
        got = p.forward_matvec(V)
        assert np.array_equal(got, p.forward_matvec(V))
    finally:
        p.close()
    rows = np.unique(np.concatenate([np.arange(0, n, 37), np.arange(n - 70, n)]))
    ref = T.matrix(X[rows], X, params) @ V.T.astype(np.float64)
    ref = ref.T + 0.3 * V[:, rows]
    err = np.linalg.norm(got[:, rows] - ref, axis=1) / np.linalg.norm(ref, axis=1)
    print("  relerr", err.max(), flush=True)
    assert err.max() <= 1e-6


@pytest.mark.parametrize("name", list(TREES))
@pytest.mark.parametrize("n,t", [(4999, 11), (5000, 5), (5121, 16), (5376, 21), (5503, 17), (6500, 5),
                                 (6657, 11), (6912, 16), (7039, 21)])
def test_products_match_oracle(name, n, t):
    mk, d = TREES[name]
    node = mk()
    rng = np.random.default_rng(n + t)
    X = rng.uniform(-2, 2, size=(n, d)).astype(np.float32)
    T = ok.TreeKernel(node.to_dict(), d)
    params = (node.to_engine_params(node.get_initial_params()) if "poly" in name
              else rng.uniform(0.8, 1.6, T.nparams)).astype(np.float32)
    print(f"tree sym {name} n={n} t={t}", flush=True)
    _run(node, T, d, X, rng.normal(size=(t, n)).astype(np.float32), params)


def test_correlation_tables_stay_one_sided():
    rng = np.random.default_rng(5)
    n, levels = 5100, 3
    X = np.stack([rng.uniform(-2, 2, n), rng.integers(0, levels, n)], axis=1).astype(np.float32)
    node = RBF(active_dims=[0]) * GD(levels, active_dims=[1])
    table = rng.uniform(0.2, 1.0, size=(levels, levels)).astype(np.float32)  # not symmetric
    T = ok.TreeKernel(node.to_dict(), 2, cat_tables=[table])
    _run(node, T, 2, X, rng.normal(size=(8, n)).astype(np.float32),
         np.array([0.8, 1.3], np.float32), table)
