"""Gradient traces of kernel trees on their generated kernel (from 5500 to 7500
points on for these trees) and on the interpreted one below, against the float64 tree restatement:
every leaf kind, isotropic and ARD, shared subtrees' adjoints, a categorical
leaf (tables need not be symmetric, so no pair is folded), ragged last blocks
and 1 .. 17 factor columns.

Bound: a term w_ab dK_ab / dtheta is formed in fp32 from a handful of
operations (<= 16 ulps with the hardware exp / sin / log), and fp32 sums run
over at most 64 terms before fp64, so |error| <= (16 + 64) 2^-24 sum |w dK|."""

import numpy as np
import pytest

from mojogp_amd import (GD, RBF, RQ, Linear, Matern12, Matern32, Matern52, Periodic, Polynomial,
                        make_ard_kernel)
from mojogp_amd._provider import NativeProvider
from oracle import kernels as ok

pytestmark = pytest.mark.gpu

TREES = {
    "rbf*per[0]+rq": (lambda: RBF() * Periodic(active_dims=[0]) + RQ(), 3),
    "ard": (lambda: make_ard_kernel((RQ(ard=True) + Matern52(ard=True))
                                    * Periodic(period=2.0, ard=True), 2), 2),
    "2*(m12+m32)*m52": (lambda: 2.0 * (Matern12() + Matern32()) * Matern52(), 5),
    "poly_ard+lin*m12_ard": (lambda: make_ard_kernel(
        Polynomial(degree=2.0, ard=True) + Linear() * Matern12(ard=True), 2), 2),
    "poly+lin_ard": (lambda: make_ard_kernel(Polynomial() + Linear(ard=True), 3), 3),
}


def _check(T, X, params, L, R, got):
    ref, mag = np.zeros(T.nparams), np.zeros(T.nparams)
    rows = np.flatnonzero(L.any(axis=0))  # the others' terms are zero
    for i in range(0, len(rows), 256):
        at = rows[i:i + 256]
        G = T.gradients(X[at], X, params)
        W = L[:, at].astype(np.float64).T @ R.astype(np.float64)
        ref += (G * W).sum(axis=(1, 2))
        mag += np.abs(G * W).sum(axis=(1, 2))
    err = np.abs(got - ref)
    print("  error / bound", np.round(err / np.maximum(80 * 2.0**-24 * mag, 1e-300), 4), flush=True)
    assert np.all(err <= 80 * 2.0**-24 * mag)


def _unused(rng, n):
    """Rows left without weight where the restatement of all would take long:
    all but 400 and the last 40."""
    return np.setdiff1d(np.arange(n - 40), rng.choice(n - 40, 400, replace=False))


@pytest.mark.parametrize("name", list(TREES))
@pytest.mark.parametrize("n,t", [(700, 17), (4095, 3), (4096, 1), (4227, 17), (7555, 17)])
def test_traces_match_oracle(name, n, t):
    mk, d = TREES[name]
    node = mk()
    rng = np.random.default_rng(n + t)
    X = rng.uniform(-2, 2, size=(n, d)).astype(np.float32)
    T = ok.TreeKernel(node.to_dict(), d)
    params = rng.uniform(0.6, 1.5, T.nparams).astype(np.float32)
    if "poly" in name:
        params = node.to_engine_params(node.get_initial_params()).astype(np.float32)
    L, R = (rng.normal(size=(t, n)).astype(np.float32) for _ in range(2))
    if n > 5000:
        L[:, _unused(rng, n)] = 0.0
    print(f"tree trace {name} n={n} t={t}", flush=True)
    p = NativeProvider(None, False, X, params, 0.2, tree_spec=node.to_tree_spec(d))
    try:
        got = p.gradient_trace(L, R)
    finally:
        p.close()
    _check(T, X, params, L, R, got)


@pytest.mark.parametrize("n", [4100, 8700])
def test_categorical_tree_is_not_folded(n):
    import ctypes as C
    from mojogp_amd import _lib
    rng = np.random.default_rng(5)
    t, levels = 6, 4
    X = np.stack([rng.uniform(-2, 2, n), rng.integers(0, levels, n)], axis=1).astype(np.float32)
    node = RBF(active_dims=[0]) * GD(levels, active_dims=[1])
    table = rng.uniform(0.2, 1.0, size=(levels, levels)).astype(np.float32)  # not symmetric
    T = ok.TreeKernel(node.to_dict(), 2, cat_tables=[table])
    params = np.array([0.8, 1.3], np.float32)
    L, R = (rng.normal(size=(t, n)).astype(np.float32) for _ in range(2))
    p = NativeProvider(None, False, X, params, 0.2, tree_spec=node.to_tree_spec(2))
    try:
        flat = np.ascontiguousarray(table.ravel())
        _lib.call("mgp_set_categorical_tables", p.handle, _lib.fptr(flat), int(flat.size))
        got = p.gradient_trace(L, R)
    finally:
        p.close()
    _check(T, X, params, L, R, got)


@pytest.mark.parametrize("n", [700, 9001])
def test_parameter_factors_are_not_rounded(n):
    """Equal points and small whole weights: every product and sum is exact in
    fp32 or fp64, so the outputscale's trace, sum W, is exact too (a factor 1 /
    outputscale rounded to fp32 would leave up to 6e-8)."""
    node = RBF() + RQ()
    rng = np.random.default_rng(n)
    X = np.tile(np.array([[0.5, -1.0]], np.float32), (n, 1))
    L, R = (rng.integers(1, 4, size=(3, n)).astype(np.float32) for _ in range(2))
    p = NativeProvider(None, False, X, np.array([0.7, 3.0, 1.1, 1.3, 7.0], np.float32), 0.2,
                       tree_spec=node.to_tree_spec(2))
    try:
        got = p.gradient_trace(L, R)
    finally:
        p.close()
    want = float((L.astype(np.float64).sum(1) * R.astype(np.float64).sum(1)).sum())
    print(f"n={n} relative", (got[[1, 4]] - want) / want, flush=True)
    if n >= 9000:  # the generated kernel
        assert np.all(np.abs(got[[1, 4]] - want) <= 1e-12 * want)
    else:
        assert np.all(np.abs(got[[1, 4]] - want) <= 16 * 2.0**-24 * want)


def test_many_parameters():
    """46 parameters: the generated kernel keeps two sums of each per lane, some
    of them in scratch memory."""
    d, n, t = 10, 4001, 5
    node = make_ard_kernel((RBF(ard=True) + RQ(ard=True)) * Periodic(period=2.0, ard=True)
                           + Matern52(ard=True), d)
    rng = np.random.default_rng(7)
    X = rng.uniform(-2, 2, size=(n, d)).astype(np.float32)
    T = ok.TreeKernel(node.to_dict(), d)
    assert T.nparams == 46
    params = rng.uniform(2.0, 5.0, T.nparams).astype(np.float32)
    L, R = (rng.normal(size=(t, n)).astype(np.float32) for _ in range(2))
    L[:, _unused(rng, n)] = 0.0
    p = NativeProvider(None, False, X, params, 0.2, tree_spec=node.to_tree_spec(d))
    try:
        got = p.gradient_trace(L, R)
    finally:
        p.close()
    _check(T, X, params, L, R, got)


def test_shared_parameter_slots():
    """Two leaves that read the same lengthscale and outputscale: no generated
    kernel, and the trace is the sum of the leaves' own."""
    n, t = 7200, 4
    rng = np.random.default_rng(11)
    X = rng.uniform(-2, 2, size=(n, 4)).astype(np.float32)
    L, R = (rng.normal(size=(t, n)).astype(np.float32) for _ in range(2))
    spec = list((RBF() + Matern52()).to_tree_spec(4))
    both = np.array([0.9, 1.3], np.float32)
    got = []
    for shared in (True, False):
        s = list(spec)
        if shared:
            assert s[1] == 4 and s[15] == 2  # parameters; the second leaf's first one
            s[1], s[15] = 2, 0
        p = NativeProvider(None, False, X, both if shared else np.tile(both, 2), 0.2, tree_spec=s)
        try:
            got.append(p.gradient_trace(L, R))
        finally:
            p.close()
    want = got[1][:2] + got[1][2:]
    mag = np.abs(L).sum() * np.abs(R).sum() / n**2  # mean |w|, up to the columns' signs
    print(got[0], want, flush=True)
    assert np.all(np.abs(got[0] - want) <= 80 * 2.0**-24 * mag * n * n)
