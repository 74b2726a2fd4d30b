"""Difference-form gradient traces (grad_pair.hip) at the edges of their
128-point blocks (odd and even block counts, ragged last block), padded input
dimensions, 1 .. 17 factor columns, isotropic and ARD, coincident points,
against the float64 oracle.

Bound: a term w_ab dK_ab is formed from a handful of fp32 operations on r^2
(<= 24 ulps with the hardware exp and sqrt, the exponent within 20 log2 e) and
fp32 sums run over at most 16 terms before fp64, so |error| <= (24 + 16) 2^-24
sum |w dK|."""

import numpy as np
import pytest

from mojogp_amd._provider import NativeProvider
from oracle import kernels as ok

pytestmark = pytest.mark.gpu

KINDS = [ok.RBF, ok.MATERN52, ok.MATERN12, ok.MATERN32]


@pytest.mark.parametrize("kind", KINDS)
@pytest.mark.parametrize("n,d,t,ard", [(1, 1, 1, False), (127, 2, 4, True), (128, 3, 5, False),
                                       (129, 7, 16, True), (384, 11, 17, True),
                                       (511, 17, 3, False), (700, 31, 11, True),
                                       (1025, 5, 33, True)])
def test_edges(monkeypatch, kind, n, d, t, ard):
    monkeypatch.setenv("MGP_GRAD_MFMA", "0")
    rng = np.random.default_rng(100 * kind + n + d)
    X = rng.normal(size=(n, d)).astype(np.float32)
    if n > 130:
        X[5] = X[130]  # coincident points: the Matern-1/2 cusp
    L, R = (rng.normal(size=(t, n)).astype(np.float32) for _ in range(2))
    ls = rng.uniform(0.7, 1.4, d if ard else 1) * np.sqrt(d)
    params = np.concatenate([ls, [1.2]]).astype(np.float32)
    print(f"kind={kind} n={n} d={d} t={t} ard={ard}", flush=True)
    p = NativeProvider(kind, ard, X, params, 0.1)
    try:
        got = p.gradient_trace(L, R)
    finally:
        p.close()
    W = L.astype(np.float64).T @ R.astype(np.float64)
    ref, mag = np.zeros(len(params)), np.zeros(len(params))
    for i in range(0, n, 256):
        G = ok.kernel_gradients(kind, X[i:i + 256], X, params, ard) * W[i:i + 256]
        ref += G.sum(axis=(1, 2))
        mag += np.abs(G).sum(axis=(1, 2))
    assert np.all(np.abs(got - ref) <= 40 * 2.0**-24 * mag + 1e-30)
