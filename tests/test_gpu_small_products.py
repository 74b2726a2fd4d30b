"""Tile products of small models and of few test points (launches whose row
tiles per wave and column splits come from the latency model): one column-tile
pair a split, splits that do not divide the pairs, row counts around a
workgroup's 128 rows and not multiples of 4 (unaligned epilogue), 1 .. 65
right-hand sides, against the float64 oracle.

Bound: the Gram-form distance carries ~2^-23 of the norm sum (<= 64 for these
inputs), i.e. at most 64 ln2 2^-24 = 2.6e-6 in an RBF value and less in the
Matern ones; the sums average it."""

import numpy as np
import pytest

from mojogp_amd._provider import NativeProvider
from oracle import kernels as ok

pytestmark = pytest.mark.gpu


def _err(a, b):
    return float(np.linalg.norm(np.asarray(a, np.float64) - b) / max(np.linalg.norm(b), 1e-30))


@pytest.mark.parametrize("n", [1, 16, 33, 127, 129, 514, 1003, 4001])
@pytest.mark.parametrize("t", [1, 7, 17, 65])
def test_square_and_cross(n, t):
    rng = np.random.default_rng(n * 100 + t)
    kind = [ok.RBF, ok.MATERN52, ok.MATERN32][(n + t) % 3]
    d = 1 + (n + t) % 12
    X = rng.normal(size=(n, d)).astype(np.float32)
    V = rng.normal(size=(t, n)).astype(np.float32)
    params = np.concatenate([rng.uniform(0.8, 1.3, d) * np.sqrt(d), [1.1]]).astype(np.float32)
    print(f"n={n} t={t} d={d} kind={kind}", flush=True)
    p = NativeProvider(kind, True, X, params, 0.1)
    try:
        got = p.forward_matvec(V)
        assert _err(got, ok.forward_matvec(kind, X, V, params, 0.1, True)) <= 2.6e-6
        for m in (1, 5, 130, 1021):
            Xs = rng.normal(size=(m, d)).astype(np.float32)
            got = p.cross_matvec(Xs, V)
            assert _err(got, ok.cross_matvec(kind, Xs, X, V, params, True)) <= 2.6e-6
    finally:
        p.close()
