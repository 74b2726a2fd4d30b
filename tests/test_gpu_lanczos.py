"""The device-side Lanczos recurrence where the Krylov space is exhausted: with
all points equal the kernel matrix has rank one, so the recurrence breaks down
(beta < 1e-10, later iterations run as no-ops) or goes on in rounding noise,
which needs its second orthogonalisation pass to stay orthogonal.

The variance at a far point is the prior's to rounding; at the point itself
it is os noise / (n os + noise) = 1e-4 at n = 5100, a difference of numbers
near 1 formed in fp32, so within 1e-5."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [600, 2000, 5100, 8000, 30000, 65536])
def test_lanczos_breakdown(n):
    from mojogp_amd._engine import load_engine, load_kernel_module
    X = np.full((n, 2), 0.5, np.float32)
    y = np.random.default_rng(0).normal(size=n).astype(np.float32)
    params = np.array([1.0, 1.0], np.float32)
    m = load_kernel_module("rbf", False, 2)
    info = m.init_provider(X, params, 0.5)
    try:
        Xs = np.array([[0.5, 0.5], [40.0, 40.0]], np.float32)
        r = load_engine().predict(info, y, Xs, params, 0.5, 0.0, 1, 100, 1e-3, 10, 50, True)
    finally:
        m.destroy_provider(info)
    assert np.all(np.isfinite(r["variance"]))
    assert abs(r["variance"][1] - 1.0) <= 1e-5
    assert abs(r["variance"][0] - 0.5 / (n + 0.5)) <= 1e-5
    assert abs(r["mean"][1]) <= 1e-5
