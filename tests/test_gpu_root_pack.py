"""Predictions from a cache (LOVE root packed once, 64-column chunks) give the
bits of predictions that pack it per call: ranks around the chunk sizes (1, 16,
17, 32, 64, one column left over, several chunks) and ragged test sets, on the tile, the difference and the
kernel-tree route (the last two ignore the packing)."""

import numpy as np
import pytest

from mojogp_amd import RBF, Matern52
from mojogp_amd._engine import load_engine, load_kernel_module

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind,n,rank", [("matern52", 700, 1), ("rbf", 1001, 16),
                                         ("matern32", 515, 17), ("matern52", 900, 64),
                                         ("rbf", 640, 65), ("matern52", 1003, 130),
                                         ("matern12", 600, 70), ("tree", 600, 40)])
def test_cache_matches_direct_prediction(kind, n, rank):
    rng = np.random.default_rng(n + rank)
    d = 3
    X = rng.normal(size=(n, d)).astype(np.float32)
    y = np.sin(X.sum(1)).astype(np.float32)
    if kind == "tree":
        node = RBF() + Matern52()
        from mojogp_amd._engine import KernelModule
        m = KernelModule(None, False, d, tree_spec=node.to_tree_spec(d))
        params = np.array([1.0, 1.1, 0.8, 0.6], np.float32)
    else:
        m = load_kernel_module(kind, False, d)
        params = np.array([1.1, 1.2], np.float32)
    eng = load_engine()
    info = m.init_provider(X, params, 0.1)
    try:
        cache = eng.prepare_prediction_cache(info, y, params, 0.1, 0.0, 1, 100, 1e-3, 10, rank,
                                             True)["cache_handle"]
        for mt in (1, 33, 400):
            Xs = rng.normal(size=(mt, d)).astype(np.float32)
            a = eng.predict_with_cache(info, cache, Xs, params, 0.1, 0.0, 1)
            b = eng.predict(info, y, Xs, params, 0.1, 0.0, 1, 100, 1e-3, 10, rank, True)
            assert np.array_equal(a["mean"], b["mean"])
            assert np.array_equal(a["variance"], b["variance"])
        eng.destroy_prediction_cache(cache)
    finally:
        m.destroy_provider(info)
