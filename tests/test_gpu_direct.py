"""Difference products (direct.hip) at the edges of their tiles: 64-column LDS
tiles, 128- or 256-row workgroups, the 1 / 4 / 16 / 64 right-hand-side forms
and every padded input dimension, against the float64 oracle; the fixed-arena
call (splits cut to what the array holds) against the allocating one.

Bound: every product term carries a kernel value within a few fp32 ulps of
r^2 and of the exponent (u <= 20 log2 e scaled by 2^-24 each), so the normwise
error stays below 2e-6 for lengthscales of the order of the data."""

import numpy as np
import pytest

from mojogp_amd._provider import NativeProvider
from oracle import kernels as ok

pytestmark = pytest.mark.gpu

KINDS = [ok.RBF, ok.MATERN52, ok.MATERN12, ok.MATERN32]


def _err(a, b):
    b = np.asarray(b, np.float64)
    return float(np.linalg.norm(np.asarray(a, np.float64) - b) / max(np.linalg.norm(b), 1e-30))


@pytest.mark.parametrize("kind", KINDS)
@pytest.mark.parametrize("n,d,t", [(1, 1, 1), (63, 2, 4), (64, 3, 5), (65, 4, 16), (257, 7, 17),
                                   (300, 9, 64), (511, 11, 65), (640, 17, 3), (1000, 31, 11),
                                   (1025, 32, 33)])
def test_edges(kind, n, d, t):
    rng = np.random.default_rng(1000 * kind + n + d)
    X = rng.normal(size=(n, d)).astype(np.float32)
    Xs = rng.normal(size=(max(1, n // 3), d)).astype(np.float32)
    V = rng.normal(size=(t, n)).astype(np.float32)
    params = np.concatenate([rng.uniform(0.7, 1.4, d) * np.sqrt(d), [1.2]]).astype(np.float32)
    print(f"kind={kind} n={n} d={d} t={t}", flush=True)
    p = NativeProvider(kind, True, X, params, 0.1)
    try:
        got = p.direct_matvec(V)
        cross = p.cross_matvec(Xs, V) if kind == ok.MATERN12 else None
    finally:
        p.close()
    assert _err(got, ok.forward_matvec(kind, X, V, params, 0.1, True)) <= 2e-6
    if cross is not None:
        assert _err(cross, ok.cross_matvec(kind, Xs, X, V, params, True)) <= 2e-6


def test_columns_are_independent():
    """A right-hand side's result does not depend on the others' values."""
    rng = np.random.default_rng(3)
    n = 700
    X = rng.normal(size=(n, 3)).astype(np.float32)
    V = rng.normal(size=(6, n)).astype(np.float32)
    W = V.copy()
    W[3] = np.inf
    p = NativeProvider(ok.MATERN12, False, X, np.array([1.0, 1.0], np.float32), 0.1)
    try:
        a, b = p.forward_matvec(V), p.forward_matvec(W)
    finally:
        p.close()
    keep = [0, 1, 2, 4, 5]
    assert np.array_equal(a[keep], b[keep])
    assert not np.isfinite(b[3]).any()


@pytest.mark.parametrize("n,t", [(2000, 11), (300001, 16)])
def test_fixed_arena(n, t):
    """mgp_forward_matvec_device_noalloc on the difference route: split
    partials inside the fixed array, none where not even two splits fit
    (300001 x 16 fp64 sums)."""
    from mojogp_amd import _lib
    from test_zz_no_alloc import _Dev, _hip
    hip = _hip()
    rng = np.random.default_rng(n)
    X = rng.normal(size=(n, 1)).astype(np.float32)
    V = rng.normal(size=(t, n)).astype(np.float32)
    src, dst = _Dev(hip, V.nbytes), _Dev(hip, V.nbytes)
    src.put(V)
    p = NativeProvider(ok.MATERN12, False, X, np.array([0.7, 1.0], np.float32), 0.1)
    try:
        _lib.call("mgp_forward_matvec_device", p.handle, src.ptr, t, dst.ptr)
        want = dst.get(V.shape)
        _lib.call("mgp_forward_matvec_device_noalloc", p.handle, src.ptr, t, dst.ptr)
        got = dst.get(V.shape)
    finally:
        p.close()
        src.free()
        dst.free()
    assert _err(got, want) <= 2e-7  # the same fp64 sums in another order, rounded once


@pytest.mark.parametrize("kind", [ok.MATERN12, ok.RBF])
@pytest.mark.parametrize("n,d,t", [(12151, 1, 5), (11264, 3, 16), (10241, 6, 70), (7296, 12, 11),
                                   (5503, 32, 7), (15105, 1, 5), (13313, 3, 16), (11265, 6, 70)])
def test_symmetric_blocks(kind, n, d, t):
    """Square products on unordered pairs: odd and even counts of 256- and
    128-point blocks, ragged last stage, a second column chunk; repeated calls
    bit for bit the same."""
    rng = np.random.default_rng(n + d)
    X = rng.normal(size=(n, d)).astype(np.float32)
    V = rng.normal(size=(t, n)).astype(np.float32)
    params = np.concatenate([rng.uniform(0.7, 1.4, d) * np.sqrt(d), [1.2]]).astype(np.float32)
    p = NativeProvider(kind, True, X, params, 0.1)
    try:
        got = p.direct_matvec(V)
        assert np.array_equal(got, p.direct_matvec(V))
    finally:
        p.close()
    rows = np.unique(np.concatenate([np.arange(0, n, 31), np.arange(n - 70, n)]))
    ref = ok.forward_matvec(kind, X, V, params, 0.1, True, rows=rows)
    assert _err(got[:, rows], ref) <= 2e-6


@pytest.mark.parametrize("kind", [ok.MATERN12, ok.MATERN52])
@pytest.mark.parametrize("n,d,t", [(3001, 1, 1), (2000, 5, 3), (3001, 1, 11), (1500, 7, 40),
                                   (15001, 1, 5), (13000, 4, 16), (6001, 24, 9)])
def test_sums_are_fp64(kind, n, d, t):
    """Right-hand sides without a common sign, on equal points: every kernel
    value is exactly 1, so what is left is the rounding of the sums.  Products
    and sums are fp64; the result is rounded once (one-sided, half an ulp), and
    on unordered pairs (the last three) the partial sums once each, whose mean
    squares add up to at most n, the result's own another n."""
    rng = np.random.default_rng(n + t)
    X = np.tile(rng.normal(size=d).astype(np.float32), (n, 1))
    V = rng.normal(size=(t, n)).astype(np.float32)
    os = np.float32(1.25)  # exact in any product below
    p = NativeProvider(kind, False, X, np.array([0.7, os], np.float32), 0.5)
    try:
        got = p.direct_matvec(V).astype(np.float64)
        cross = p.cross_matvec(X[:70], V) if kind == ok.MATERN12 else None
    finally:
        p.close()
    V = V.astype(np.float64)
    want = 1.25 * V.sum(axis=1, keepdims=True)
    ulp = 2.0**-24 * (1 + 1e-6)
    if cross is not None:
        assert np.all(np.abs(cross - want) <= ulp * np.abs(want))
    want = want + 0.5 * V
    if n < 5500:
        assert np.all(np.abs(got - want) <= ulp * np.abs(want))
    else:
        assert np.sqrt(np.mean((got - want) ** 2)) <= 1.25 * 2.0**-24 * np.sqrt(2.0 * n)


@pytest.mark.parametrize("t", [17, 32, 33, 48, 49])
def test_unused_column_groups(t):
    """A product of 17 to 63 columns skips the 16-column groups it does not
    fill: the same bits as the first columns of a full one."""
    rng = np.random.default_rng(t)
    n = 1333
    X = rng.normal(size=(n, 3)).astype(np.float32)
    V = rng.normal(size=(64, n)).astype(np.float32)
    p = NativeProvider(ok.MATERN12, False, X, np.array([0.9, 1.1], np.float32), 0.1)
    try:
        assert np.array_equal(p.forward_matvec(V[:t]), p.forward_matvec(V)[:t])
    finally:
        p.close()


@pytest.mark.parametrize("n,d,t", [(19999, 2, 20), (20000, 16, 17), (20003, 3, 32), (20001, 17, 24),
                                   (20000, 1, 33)])
def test_two_symmetric_passes(n, d, t):
    """17 to 32 columns around the line where they run as two symmetric passes."""
    rng = np.random.default_rng(n + t)
    X = rng.normal(size=(n, d)).astype(np.float32)
    V = rng.normal(size=(t, n)).astype(np.float32)
    params = np.concatenate([rng.uniform(0.7, 1.4, d) * np.sqrt(d), [1.2]]).astype(np.float32)
    p = NativeProvider(ok.MATERN12, True, X, params, 0.1)
    try:
        got = p.forward_matvec(V)
    finally:
        p.close()
    rows = np.unique(np.concatenate([np.arange(0, n, 61), np.arange(n - 70, n)]))
    assert _err(got[:, rows], ok.forward_matvec(ok.MATERN12, X, V, params, 0.1, True, rows=rows)) <= 2e-6
