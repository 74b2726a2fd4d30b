"""Symmetric products whose partial sums do not fit what is left of the device's
memory run on their one-sided kernel, which needs little, with its results to
the bit; the next product with memory at hand is symmetric again."""

import ctypes as C

import numpy as np
import pytest

from mojogp_amd import RBF, RQ, Periodic
from mojogp_amd._provider import NativeProvider
from oracle import kernels as ok
from test_zz_no_alloc import _Dev, _hip

pytestmark = pytest.mark.gpu

LEFT = 3 << 29  # 1.5 GiB (the allocation is rounded: up to 2 GiB are left)


# partial sums of n^2 / 8 and n^2 / 128 bytes: 2.8 GB
CASES = (("tree", 150_000, 7), ("difference", 150_000, 7), ("one column", 600_000, 1))


def _provider(route, X):
    if route == "tree":
        spec = (RBF() * Periodic(active_dims=[0]) + RQ()).to_tree_spec(1)
        return NativeProvider(None, False, X, np.linspace(0.9, 1.4, 8).astype(np.float32), 0.1,
                              tree_spec=spec)
    return NativeProvider(ok.MATERN12 if route == "difference" else ok.MATERN52, False, X,
                          np.array([0.8, 1.2], np.float32), 0.1)


def test_falls_back(monkeypatch):
    hip = _hip()  # (the runtime that the library runs on)
    held = []
    for route, n, t in CASES:
        rng = np.random.default_rng(n)
        X = rng.normal(size=(n, 1)).astype(np.float32)
        held.append((route, _provider(route, X), rng.normal(size=(t, n)).astype(np.float32)))
    try:
        monkeypatch.setenv("MGP_SYM_MATVEC", "0")
        one = [p.forward_matvec(V) for _, p, V in held]
        monkeypatch.delenv("MGP_SYM_MATVEC")
        free, total = C.c_size_t(), C.c_size_t()
        assert hip.hipDeviceSynchronize() == 0
        assert hip.hipMemGetInfo(C.byref(free), C.byref(total)) == 0
        hold = _Dev(hip, free.value - LEFT)
        got = []
        try:
            for route, p, V in held:
                print(route, flush=True)
                got.append(p.forward_matvec(V))
        finally:
            hold.free()
        sym = [p.forward_matvec(V) for _, p, V in held]
    finally:
        for _, p, _ in held:
            p.close()
    for a, g, s in zip(one, got, sym):
        assert np.array_equal(g, a)
        assert not np.array_equal(s, a)
        assert np.linalg.norm(s - a) <= 2e-6 * np.linalg.norm(a)
