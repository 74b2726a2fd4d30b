"""Device memory that predictions leave behind: the LOVE variance's [rank][m]
block of a large test set is given back."""

import ctypes as C

import numpy as np
import pytest

from mojogp_amd._engine import load_engine, load_kernel_module
from test_zz_no_alloc import _hip

pytestmark = pytest.mark.gpu


def _free():
    hip = _hip()
    free, total = C.c_size_t(), C.c_size_t()
    assert hip.hipDeviceSynchronize() == 0
    assert hip.hipMemGetInfo(C.byref(free), C.byref(total)) == 0
    return free.value


def _cache(kind, n, rank):
    rng = np.random.default_rng(n)
    X = rng.normal(size=(n, 1)).astype(np.float32)
    y = np.sin(3 * X[:, 0]).astype(np.float32)
    params = np.array([0.7, 1.0], np.float32)
    m = load_kernel_module(kind, False, 1)
    info = m.init_provider(X, params, 0.1)
    cache = load_engine().prepare_prediction_cache(info, y, params, 0.1, 0.0, 1, 100, 1e-3, 10, rank,
                                                   True, y)["cache_handle"]
    return m, info, cache, params


def test_large_test_set_is_not_kept():
    rank, points = 200, 300_000  # a block of 240 MB; the packed test points take ~45 MB
    m, info, cache, params = _cache("matern52", 600, rank)
    eng = load_engine()
    Xs = np.linspace(-3, 3, points, dtype=np.float32)[:, None]
    try:
        small = eng.predict_with_cache(info, cache, Xs[::1000], params, 0.1, 0.0, 1)
        before = _free()
        large = eng.predict_with_cache(info, cache, Xs, params, 0.1, 0.0, 1)
        assert before - _free() < 120e6
        again = eng.predict_with_cache(info, cache, Xs[::1000], params, 0.1, 0.0, 1)
    finally:
        eng.destroy_prediction_cache(cache)
        m.destroy_provider(info)
    assert np.array_equal(small["variance"], again["variance"])
    assert np.abs(large["variance"][::1000] - small["variance"]).max() <= 1e-5


@pytest.mark.parametrize("kind,copies", [("matern52", 2), ("matern12", 1)])
def test_root_is_packed_where_it_is_read(kind, copies):
    """A cache holds alpha, the root and, where predictions take the tile route,
    the root's packing (the difference products never read one)."""
    n, rank = 100_000, 64  # the root: 26 MB
    m, info, cache, params = _cache(kind, n, rank)
    try:
        held = -_free()
        load_engine().destroy_prediction_cache(cache)
        held += _free()
    finally:
        m.destroy_provider(info)
    print(kind, held / (4.0 * n * rank), "roots", flush=True)
    assert copies * 0.9 <= held / (4.0 * n * rank) <= copies + 0.2
