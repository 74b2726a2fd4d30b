"""Symmetric products with one and two right-hand sides (k_sym_vec): 1 .. 7
blocks of 256 points (odd and even counts, a last block of one point), every
count of distance MFMAs, both column counts bit for bit the same per column,
and the automatic route from 5000 points on.

Bound: as for the tile products, a Gram-form distance error of ~2^-23 of the
norm sum (<= 64 here) gives at most 64 ln2 2^-24 = 2.6e-6 per value."""

import numpy as np
import pytest

from mojogp_amd._provider import NativeProvider
from oracle import kernels as ok

pytestmark = pytest.mark.gpu


def _err(a, b):
    return float(np.linalg.norm(np.asarray(a, np.float64) - b) / max(np.linalg.norm(b), 1e-30))


def _check(kind, n, d, seed):
    rng = np.random.default_rng(seed)
    X = rng.normal(size=(n, d)).astype(np.float32)
    V = rng.normal(size=(2, n)).astype(np.float32)
    params = np.concatenate([rng.uniform(0.8, 1.3, d) * np.sqrt(d), [1.1]]).astype(np.float32)
    p = NativeProvider(kind, True, X, params, 0.1)
    try:
        two = p.forward_matvec(V)
        one = [p.forward_matvec(V[c]) for c in range(2)]
        again = p.forward_matvec(V)
    finally:
        p.close()
    assert np.array_equal(two, again)
    assert np.array_equal(two[0], one[0]) and np.array_equal(two[1], one[1])
    rows = np.unique(np.concatenate([np.arange(0, n, max(1, n // 400)), [n - 1]]))
    ref = ok.forward_matvec(kind, X, V, params, 0.1, True, rows=rows)
    assert _err(two[:, rows], ref) <= 2.6e-6


@pytest.mark.parametrize("kind", [ok.RBF, ok.MATERN52, ok.MATERN32])
@pytest.mark.parametrize("n,d", [(1, 1), (255, 2), (257, 8), (512, 9), (769, 20), (1024, 30),
                                 (1537, 4)])
def test_forced_edges(monkeypatch, kind, n, d):
    monkeypatch.setenv("MGP_SYM_MATVEC", "1")
    print(f"kind={kind} n={n} d={d}", flush=True)
    _check(kind, n, d, n + d)


@pytest.mark.parametrize("kind,n,d", [(ok.MATERN52, 5003, 3), (ok.RBF, 8193, 16)])
def test_automatic_route(kind, n, d):
    print(f"kind={kind} n={n} d={d}", flush=True)
    _check(kind, n, d, n)
