"""MGP_SYM_MATVEC on the products formed per pair (differences, kernel trees):
0 keeps the one-sided kernel at any size, 1 takes the symmetric one at any
size, and the two agree over the sizes where blocks, stages and right-hand
sides run out (one point, a stage of 64, a block of 128 or 256, even and odd
block counts, 1 .. 16 columns and a second chunk).

Both sum the same kernel values (bit for bit: the same instructions on the
same coordinates).  Differences: fp64 sums, so they part by the fp32 roundings
of the partial sums, at most a few per entry.  Trees: fp32 sums over at most
128 terms before fp64."""

import numpy as np
import pytest

from mojogp_amd import RBF, RQ, Linear, Matern52, Periodic, Polynomial, make_ard_kernel
from mojogp_amd._provider import NativeProvider
from oracle import kernels as ok

pytestmark = pytest.mark.gpu

TREES = {"rbf*per[0]+rq": (lambda: RBF() * Periodic(active_dims=[0]) + RQ(), 3),
         "poly+lin": (lambda: Polynomial(degree=2.0) + Linear(), 5)}


def _both(monkeypatch, p, V):
    out = []
    for mode in ("0", "1"):
        monkeypatch.setenv("MGP_SYM_MATVEC", mode)
        out.append(p.forward_matvec(V).astype(np.float64))
    monkeypatch.delenv("MGP_SYM_MATVEC")
    return out + [p.forward_matvec(V).astype(np.float64)]


def _rms(a, b):
    return np.sqrt(np.mean((a - b) ** 2) / np.mean(b ** 2))


@pytest.mark.parametrize("n,t", [(1, 1), (63, 16), (64, 4), (65, 5), (129, 11), (256, 17), (257, 2),
                                 (700, 16), (1153, 7)])
@pytest.mark.parametrize("d", [1, 5, 12])
def test_difference_products(monkeypatch, d, n, t):
    rng = np.random.default_rng(n + d)
    X = rng.normal(size=(n, d)).astype(np.float32)
    V = rng.normal(size=(t, n)).astype(np.float32)
    print(f"d={d} n={n} t={t}", flush=True)
    p = NativeProvider(ok.MATERN12, True, X,
                       np.array([1.0 + 0.1 * k for k in range(d)] + [1.25], np.float32), 0.25)
    try:
        one, sym, auto = _both(monkeypatch, p, V)
    finally:
        p.close()
    assert np.array_equal(one, auto)  # small products stay one-sided
    assert _rms(sym, one) <= 4 * 2.0**-24 + 2.0**-24 * np.sqrt(n)  # the last: cancelled sums
    if n >= 700:
        assert not np.array_equal(one, sym)


@pytest.mark.parametrize("n,t", [(1, 1), (64, 16), (65, 3), (255, 11), (257, 5), (513, 17),
                                 (1100, 16)])
@pytest.mark.parametrize("name", list(TREES))
def test_tree_products(monkeypatch, name, n, t):
    mk, d = TREES[name]
    node = mk()
    rng = np.random.default_rng(n + t)
    X = rng.uniform(-1, 1, size=(n, d)).astype(np.float32)
    V = rng.normal(size=(t, n)).astype(np.float32)
    params = node.to_engine_params(node.get_initial_params()).astype(np.float32)
    print(f"{name} n={n} t={t}", flush=True)
    p = NativeProvider(None, False, X, params, 0.25, tree_spec=node.to_tree_spec(d))
    try:
        one, sym, auto = _both(monkeypatch, p, V)
    finally:
        p.close()
    assert np.array_equal(one, auto)
    assert _rms(sym, one) <= 2.0**-24 * (16 + np.sqrt(n))
    if n >= 1100:
        assert not np.array_equal(one, sym)


@pytest.mark.parametrize("kind", ["difference", "tree"])
def test_off_above_the_automatic_line(monkeypatch, kind):
    rng = np.random.default_rng(3)
    n, t = 16000, 8  # the lines at d = 2: 14000 for the differences, less for the tree
    X = rng.normal(size=(n, 2)).astype(np.float32)
    V = rng.normal(size=(t, n)).astype(np.float32)
    if kind == "tree":
        node = RBF() * Periodic(active_dims=[0]) + RQ()
        p = NativeProvider(None, False, X, np.linspace(0.9, 1.4, 8).astype(np.float32), 0.1,
                           tree_spec=node.to_tree_spec(2))
    else:
        p = NativeProvider(ok.MATERN12, False, X, np.array([1.0, 1.0], np.float32), 0.1)
    try:
        one, sym, auto = _both(monkeypatch, p, V)
    finally:
        p.close()
    assert np.array_equal(sym, auto) and not np.array_equal(one, sym)
    assert _rms(sym, one) <= 2e-6


@pytest.mark.parametrize("n", [900, 4999, 5000])
def test_costly_trees_have_a_smallest_size(monkeypatch, n):
    """The dearer a tree's values the earlier it goes symmetric, but not below 5000
    points, where blocks are too few."""
    d = 10
    node = make_ard_kernel((RBF(ard=True) + RQ(ard=True)) * Periodic(period=2.0, ard=True)
                           + Matern52(ard=True), d)
    rng = np.random.default_rng(n)
    X = rng.uniform(-1, 1, size=(n, d)).astype(np.float32)
    params = rng.uniform(2.0, 5.0, 46).astype(np.float32)
    p = NativeProvider(None, False, X, params, 0.1, tree_spec=node.to_tree_spec(d))
    try:
        one, sym, auto = _both(monkeypatch, p, rng.normal(size=(6, n)).astype(np.float32))
    finally:
        p.close()
    assert np.array_equal(auto, one if n < 5000 else sym)


@pytest.mark.parametrize("bad", [np.inf, np.nan])
@pytest.mark.parametrize("route,n,t", [("difference", 700, 7), ("tree", 700, 16), ("one", 700, 1),
                                       ("two", 5003, 2)])
def test_one_bad_entry_stays_in_its_column(monkeypatch, route, n, t, bad):
    """An infinity or NaN in a right-hand side: its column is not finite where the
    one-sided kernel's is not, the other columns keep their bits."""
    rng = np.random.default_rng(n + t)
    X = rng.uniform(-1, 1, size=(n, 2)).astype(np.float32)
    V = rng.normal(size=(t, n)).astype(np.float32)
    if route == "tree":
        node = RBF() * Periodic(active_dims=[0]) + RQ()
        p = NativeProvider(None, False, X, np.linspace(0.9, 1.4, 8).astype(np.float32), 0.1,
                           tree_spec=node.to_tree_spec(2))
    else:
        kind = ok.MATERN12 if route == "difference" else ok.MATERN52
        p = NativeProvider(kind, False, X, np.array([1.0, 1.0], np.float32), 0.1)
    W = V.copy()
    W[t - 1, n // 3] = bad
    try:
        _, clean, _ = _both(monkeypatch, p, V)
        one, sym, _ = _both(monkeypatch, p, W)
    finally:
        p.close()
    assert np.array_equal(clean[:t - 1], sym[:t - 1])
    assert np.array_equal(np.isfinite(one[t - 1]), np.isfinite(sym[t - 1]))
    assert not np.isfinite(sym[t - 1]).any()
