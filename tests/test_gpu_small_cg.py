"""The two-launch CG iteration of small unpreconditioned systems against the
general one (the symmetric product forced by MGP_SYM_MATVEC=1 takes the
separate vector kernels): edges of the quads a thread carries (4096 points) and
of the route (7000; larger sizes run the separate kernels on both sides), ragged
sizes, 1 .. 16 columns, a noise vector, and the oracle's solve at convergence.

Three iterations of the same recurrence on products that agree to ~2e-7:
alpha and beta are ratios of inner products perturbed by ~1e-6, and more
iterations would only show fp32 CG's own loss of orthogonality (unconverged
solutions of two correct paths then part by 1e-4 and more).  nll, the
quadratic form and the log determinant within 2e-5; the gradient, a difference
of two traces several times its size, within the 1e-3 that the engine's
gradients are held to.
"""

import ctypes as C
import os

import numpy as np
import pytest

from mojogp_amd import _lib
from mojogp_amd._provider import NativeProvider
from oracle import kernels as ok

pytestmark = pytest.mark.gpu


def _bbmm(p, y, probes, iters, general):
    old = os.environ.get("MGP_SYM_MATVEC")
    if general:
        os.environ["MGP_SYM_MATVEC"] = "1"
    try:
        g = np.zeros(p.nparams + 1, np.float32)
        nll, iq, ld, pl = (C.c_float() for _ in range(4))
        ci, ms = C.c_int(), C.c_double()
        _lib.call("mgp_bbmm_eval", p.handle, _lib.fptr(y), 0.1, probes, iters, iters, 0.0, 3, 0,
                  C.byref(nll), C.byref(iq), C.byref(ld), _lib.fptr(g), C.byref(ci), C.byref(pl),
                  C.byref(ms))
    finally:
        if old is None:
            os.environ.pop("MGP_SYM_MATVEC", None)
        else:
            os.environ["MGP_SYM_MATVEC"] = old
    return np.array([nll.value, iq.value, ld.value]), g, ci.value


@pytest.mark.parametrize("n,probes,vec", [(5, 3, False), (63, 0, False), (1001, 15, True),
                                          (4096, 10, False), (4097, 10, True), (8193, 4, False),
                                          (16384, 10, False), (16381, 0, True),
                                          (16385, 2, False), (6999, 15, True), (7000, 3, False),
                                          (7001, 10, False)])
def test_iterations_match_the_general_path(n, probes, vec):
    rng = np.random.default_rng(n)
    d = 3
    X = rng.normal(size=(n, d)).astype(np.float32)
    y = rng.normal(size=n).astype(np.float32)
    params = np.array([0.9, 1.1, 1.3, 1.2], np.float32)
    p = NativeProvider(ok.MATERN52, True, X, params, 2.0)
    try:
        if vec:
            p.set_noise_vector(rng.uniform(1.0, 3.0, n).astype(np.float32))
        print(f"n={n} probes={probes} vec={vec}", flush=True)
        a, ga, ia = _bbmm(p, y, probes, 3, False)
        b, gb, ib = _bbmm(p, y, probes, 3, True)
    finally:
        p.close()
    assert ia == ib
    assert np.allclose(a, b, rtol=2e-5, atol=2e-5 * np.abs(b).max())
    assert np.linalg.norm(ga - gb) <= 1e-3 * np.linalg.norm(gb)


def test_converged_quadratic_form():
    rng = np.random.default_rng(2)
    n = 1203
    X = rng.normal(size=(n, 2)).astype(np.float32)
    y = rng.normal(size=n).astype(np.float32)
    params = np.array([0.7, 1.1], np.float32)
    p = NativeProvider(ok.RBF, False, X, params, 0.5)
    try:
        a, _, _ = _bbmm(p, y, 4, 200, False)
    finally:
        p.close()
    K = ok.kernel_matrix(ok.RBF, X, X, params, False) + 0.5 * np.eye(n)
    yc = y.astype(np.float64) - np.float32(0.1)
    want = yc @ np.linalg.solve(K, yc)
    assert abs(a[1] - want) <= 2e-5 * want


@pytest.mark.parametrize("n", [777, 4500])
def test_column_without_a_direction(n):
    """Targets equal to the mean leave the first column zero: p.Ap = 0, so it
    keeps x = 0 (no step, no NaN) while the probes go on, as on the general path."""
    rng = np.random.default_rng(n)
    X = rng.normal(size=(n, 2)).astype(np.float32)
    y = np.full(n, np.float32(0.1))
    p = NativeProvider(ok.RBF, False, X, np.array([0.8, 1.1], np.float32), 0.4)
    try:
        a, ga, ia = _bbmm(p, y, 6, 4, False)
        b, gb, ib = _bbmm(p, y, 6, 4, True)
    finally:
        p.close()
    assert ia == ib and a[1] == 0.0 and b[1] == 0.0
    assert np.isfinite(a).all() and np.isfinite(ga).all()
    assert np.allclose(a, b, rtol=2e-5)
    assert np.linalg.norm(ga - gb) <= 1e-3 * np.linalg.norm(gb)


def test_columns_that_stop_moving():
    """A system solved to rounding long before the last iteration: residuals reach
    the noise floor, where steps are skipped or shrink, and the solution stays."""
    rng = np.random.default_rng(8)
    n = 900
    X = rng.normal(size=(n, 1)).astype(np.float32)
    y = rng.normal(size=n).astype(np.float32)
    p = NativeProvider(ok.RBF, False, X, np.array([0.6, 1.0], np.float32), 2.0)
    try:
        a, ga, _ = _bbmm(p, y, 5, 40, False)
        b, gb, _ = _bbmm(p, y, 5, 400, False)
    finally:
        p.close()
    assert np.isfinite(b).all() and np.isfinite(gb).all()
    assert abs(a[1] - b[1]) <= 2e-5 * abs(a[1])
