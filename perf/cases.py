"""The work whose speed and accuracy this framework is measured by.

Every case goes through an entry point that a program calls: the kernel-matrix
products and gradient traces of a provider, the prediction engine, the LMC
product and a whole fit.  Device arrays are torch tensors (handed over by
address); host arrays where the entry point takes host data.  The sizes are
those of bench.py's configurations, of the tests, and of the range between
them: a few hundred points up to 250 000, 1 to 16 input dimensions, 1 to 16
right-hand sides (1 + 10 probes is the training default) and 64 for LMC.
"""

import ctypes as C
import math

import numpy as np
import torch

from mojogp_amd import RBF, RQ, Matern12, Matern32, Matern52, Periodic, SingleOutputGP, _lib
from mojogp_amd._engine import load_engine, load_kernel_module
from mojogp_amd._provider import NativeProvider
from mojogp_amd.kernel import make_ard_kernel

LEAVES = {"rbf": RBF, "matern12": Matern12, "matern32": Matern32, "matern52": Matern52}
TREES = ("rbf+matern52", "seasonal")
# floating-point operations of one kernel value beside its distance, and the
# number of exp / sqrt / sin / log it takes (counted as one each)
VALUE_FLOPS = {"rbf": 6, "matern12": 6, "matern32": 9, "matern52": 11, "rbf+matern52": 20,
               "seasonal": 28}


def listed():
    return [
        # one product of a small model: latency of a call, one right-hand side
        # (the solve for alpha and the Lanczos root are made of such calls)
        {"name": "product-small", "op": "product", "kernel": "rbf", "ard": False, "n": 1000,
         "d": 2, "t": 1, "ls": 1.0, "dense": False},
        # one training product of a middle-sized model (y and 10 probes), odd n
        {"name": "product-mid", "op": "product", "kernel": "matern52", "ard": True, "n": 12007,
         "d": 6, "t": 11, "ls": 1.0, "dense": False},
        # the benchmark's product (y and 15 probes at N = 250 000)
        {"name": "product-large", "op": "product", "kernel": "matern52", "ard": True,
         "n": 250000, "d": 16, "t": 16, "ls": 1.0, "dense": False},
        # Matern-1/2, whose distances are never taken in Gram form
        {"name": "product-matern12", "op": "product", "kernel": "matern12", "ard": True,
         "n": 20011, "d": 5, "t": 11, "ls": 1.0, "dense": False},
        # the materialized route's product at the benchmark's size
        {"name": "product-dense", "op": "product", "kernel": "rbf", "ard": False, "n": 40000,
         "d": 4, "t": 16, "ls": 1.5, "dense": True},
        # a composite kernel (trend with a season, plus a rough part)
        {"name": "product-tree", "op": "product", "kernel": "seasonal", "ard": False, "n": 20000,
         "d": 4, "t": 11, "ls": 1.0, "dense": False},
        # the gradient step of training: every parameter's trace, 16 weight columns
        {"name": "trace", "op": "trace", "kernel": "matern52", "ard": True, "n": 50000, "d": 8,
         "t": 16, "ls": 1.0},
        # the same of a composite kernel, with the default number of probes
        {"name": "trace-tree", "op": "trace", "kernel": "seasonal", "ard": False, "n": 10007,
         "d": 4, "t": 11, "ls": 1.0},
        # a whole fit of a small model (config 1's size), 10 Adam steps
        {"name": "fit-small", "op": "fit", "kernel": "rbf", "ard": False, "n": 2000, "d": 1,
         "steps": 10},
        # the first prediction after a fit: alpha, the LOVE root, mean and variance
        {"name": "predict", "op": "predict", "kernel": "matern52", "ard": False, "n": 20000,
         "d": 4, "m": 1000, "ls": 0.7},
        # a later one from the prediction cache (serving)
        {"name": "serve", "op": "serve", "kernel": "matern52", "ard": True, "n": 20000, "d": 6,
         "m": 500, "ls": 1.0},
        # the multi-output product, two latents and four tasks
        {"name": "lmc", "op": "lmc", "n": 20000, "d": 6, "t": 11, "tasks": 4},
    ]


def _log(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def draw(rng):
    op = rng.choice(["product"] * 6 + ["trace"] * 3 + ["serve"] * 2 + ["predict", "fit", "lmc"])
    ls = round(_log(rng, 0.3, 2.0), 3)
    d = rng.randint(1, 16)
    if op in ("product", "trace"):
        kernel = rng.choice(sorted(LEAVES) + sorted(TREES))
        tree = kernel in TREES
        # the per-pair kernels (and what may take them) stop earlier: their
        # cost stays below the largest listed case
        hi = 12000 if tree and op == "trace" else 25000 if tree or op == "trace" else 40000
        case = {"op": op, "kernel": kernel, "ard": not tree and rng.random() < 0.6,
                "n": int(_log(rng, 300, hi)), "d": min(d, 6) if tree else d,
                "t": rng.choice([1, 6, 11, 11, 16, rng.randint(2, 16)]), "ls": ls}
        if op == "product":
            case["dense"] = not tree and rng.random() < 0.25
            if not tree and rng.random() < 0.15:
                case["t"] = rng.randint(17, 64)
        return case
    if op == "fit":
        return {"op": op, "kernel": rng.choice(["rbf", "matern32", "matern52"]),
                "ard": rng.random() < 0.5, "n": int(_log(rng, 300, 3000)), "d": rng.randint(1, 6),
                "steps": rng.randint(3, 8)}
    if op == "lmc":
        return {"op": op, "n": int(_log(rng, 1000, 20000)), "d": rng.randint(1, 8),
                "t": rng.choice([1, 6, 11, 16]), "tasks": rng.randint(2, 4)}
    return {"op": op, "kernel": rng.choice(["rbf", "matern32", "matern52"]),
            "ard": rng.random() < 0.5, "n": int(_log(rng, 1000, 20000)), "d": rng.randint(1, 8),
            "m": int(_log(rng, 10, 2000)), "ls": round(_log(rng, 0.6, 2.0), 3)}


# ---------------------------------------------------------------- kernels

NOISE = 0.1


def _node(case):
    if case["kernel"] == "rbf+matern52":
        return RBF() + Matern52()
    if case["kernel"] == "seasonal":
        return RBF() * Periodic(active_dims=[0]) + RQ()
    node = LEAVES[case["kernel"]](ard=case["ard"])
    return make_ard_kernel(node, case["d"]) if case["ard"] else node


def _params(case, rng):
    """Engine parameters: lengthscales around `ls` times sqrt(d) / 2 (so that
    typical distances stay a few lengthscales in any dimension), outputscale 1.1."""
    base = case["ls"] * max(1.0, math.sqrt(case["d"]) / 2)
    if case["kernel"] == "rbf+matern52":
        p = [base, 1.1, 0.6 * base, 0.5]
    elif case["kernel"] == "seasonal":  # RBF l, os; Periodic l, period, os; RQ l, alpha, os
        p = [1.5 * base, 1.1, 1.2, 1.7, 0.9, 0.8 * base, 1.3, 0.6]
    elif case["ard"]:
        p = [*(base * rng.uniform(0.8, 1.25, size=case["d"])), 1.1]
    else:
        p = [base, 1.1]
    return np.asarray(p, np.float32)


def _radial(kind, r2, os, ard):
    if kind == "rbf":
        return os * torch.exp(-0.5 * r2)
    r = torch.sqrt(r2 + 1e-20)
    if kind == "matern12":
        return os * torch.exp(torch.clamp(-r, min=-20.0) if ard else -r)
    if kind == "matern32":
        u = math.sqrt(3.0) * r
        return os * (1.0 + u) * torch.exp(torch.clamp(-u, min=-20.0))
    u = math.sqrt(5.0) * r
    return os * (1.0 + u + u * u / 3.0) * torch.exp(torch.clamp(-u, min=-20.0))


def _block(case, A, B, p):
    """K(A, B) in the arrays' type; p may require gradients."""
    def r2(ls):
        out = torch.zeros((A.shape[0], B.shape[0]), dtype=A.dtype, device=A.device)
        for k in range(A.shape[1]):
            u = (A[:, k] / ls[k])[:, None] - (B[:, k] / ls[k])[None, :]
            out = torch.addcmul(out, u, u)
        return out

    d, kind = A.shape[1], case["kernel"]
    if kind == "rbf+matern52":
        return (_radial("rbf", r2([p[0]] * d), p[1], False)
                + _radial("matern52", r2([p[2]] * d), p[3], False))
    if kind == "seasonal":
        s = torch.sin(math.pi * (A[:, 0, None] - B[None, :, 0]) / p[3]) ** 2 / p[2]
        rq = p[7] * (1.0 + r2([p[5]] * d) / (2.0 * p[6])) ** -p[6]
        return _radial("rbf", r2([p[0]] * d), p[1], False) * p[4] * torch.exp(-2.0 * s) + rq
    ls = [p[k] for k in range(d)] if case["ard"] else [p[0]] * d
    return _radial(kind, r2(ls), p[-1], case["ard"])


def _dev64(a):
    return torch.as_tensor(a).to("cuda", torch.float64)


def _rows(n):
    return max(16, (1 << 25) // max(n, 1))


def _matvec64(case, A, B, p, V):
    """K(A, B) V^T for V [t, n] in 64 bits: [t, m]."""
    step = _rows(B.shape[0])
    return torch.cat([V @ _block(case, A[i:i + step], B, p).T
                      for i in range(0, A.shape[0], step)], dim=1)


def _solve64(case, X, p, b, iterations):
    """CG in 64 bits on the dense K + NOISE I."""
    K = torch.cat([_block(case, X[i:i + _rows(X.shape[0])], X, p)
                   for i in range(0, X.shape[0], _rows(X.shape[0]))])
    x = torch.zeros_like(b)
    r = b.clone()
    q = r.clone()
    rr = r @ r
    for _ in range(iterations):
        Kq = K @ q + NOISE * q
        a = rr / (q @ Kq)
        x += a * q
        r -= a * Kq
        new = r @ r
        q = r + (new / rr) * q
        rr = new
    return x


# ---------------------------------------------------------------- inputs

def _rng(seed):
    return np.random.default_rng([20260, int(seed)])


def _points(rng, n, d):
    """Standardised features, as a program feeds them in."""
    return rng.standard_normal((n, d), dtype=np.float32)


def _targets(rng, X):
    w = rng.standard_normal((X.shape[1], 3)) / math.sqrt(X.shape[1])
    f = np.sin(1.5 * X @ w + rng.uniform(0, 6, size=3)).sum(axis=1)
    return (f + math.sqrt(NOISE) * rng.standard_normal(X.shape[0])).astype(np.float32)


def _inputs(case, seed):
    """The host arrays of a case, from the seed alone."""
    rng = _rng(seed)
    op, n, d = case["op"], case["n"], case["d"]
    X = _points(rng, n, d)
    if op == "fit":
        return {"X": X, "y": _targets(rng, X)}
    if op == "lmc":
        T = case["tasks"]
        W = rng.standard_normal((2, T, 2)) / math.sqrt(2)
        A = np.einsum("stq,suq->stu", W, W) + 0.1 * np.eye(T)
        return {"X": X, "p": [np.array([0.6 * math.sqrt(d), 1.0], np.float32),
                              np.array([1.0 * math.sqrt(d), 1.0], np.float32)],
                "A": A.astype(np.float32), "noise": rng.uniform(0.01, 0.1, T).astype(np.float32),
                "V": rng.standard_normal((case["t"], T * n), dtype=np.float32)}
    p = _params(case, rng)
    if op == "product":
        # right-hand sides of a solver: normalised, of mixed smooth and rough parts
        V = rng.standard_normal((case["t"], n), dtype=np.float32)
        V[0] = _targets(rng, X)
        V /= np.linalg.norm(V, axis=1, keepdims=True)
        return {"X": X, "p": p, "V": V}
    if op == "trace":
        # [alpha | probes] against [-alpha / 2 | K^-1 probes / (2 T)]: solves
        # leave the probes' rough part, divided by the noise
        R = rng.standard_normal((case["t"], n), dtype=np.float32)
        L = (R + 0.5 * rng.standard_normal((case["t"], n), dtype=np.float32)) / np.float32(NOISE)
        L *= np.float32(0.5 / case["t"])
        return {"X": X, "p": p, "L": L, "R": R}
    Xs = _points(rng, case["m"], d)
    return {"X": X, "p": p, "y": _targets(rng, X), "Xs": Xs}


class _State(dict):
    """What a program holds: providers and caches are given back at its end."""

    def __del__(self):
        try:
            if self.get("cache"):
                load_engine().destroy_prediction_cache(self["cache"])
            for prov in self.get("provs", ()):
                prov.close()
        except Exception:
            pass


def _provider(case, X, p):
    node = _node(case)
    spec = node.to_tree_spec(case["d"]) if case["kernel"] in TREES else None
    kind = None if spec is not None else case["kernel"]
    return NativeProvider(kind, case["ard"], X, p, NOISE, tree_spec=spec)


def prepare(case, seed):
    a = _inputs(case, seed)
    s = _State(case=case, **a)
    op = case["op"]
    if op == "product":
        s["provs"] = [_provider(case, a["X"], a["p"])]
        if case["dense"]:
            s["provs"][0].materialize()
        s["V"] = torch.from_numpy(a["V"]).cuda()
        s["out"] = torch.empty_like(s["V"])
        torch.cuda.synchronize()
    elif op == "trace":
        s["provs"] = [_provider(case, a["X"], a["p"])]
    elif op == "lmc":
        s["provs"] = [NativeProvider("rbf", False, a["X"], a["p"][0], 0.0),
                      NativeProvider("matern52", False, a["X"], a["p"][1], 0.0)]
    elif op in ("predict", "serve"):
        module = load_kernel_module(case["kernel"], case["ard"], case["d"])
        s["info"] = module.init_provider(a["X"], a["p"], NOISE)
        s["provs"] = [s["info"]["_provider"]]
        s["mean"] = float(a["y"].mean())
        if op == "serve":
            s["alpha"] = _alpha(case, a, 100)
            s["cache"] = load_engine().prepare_prediction_cache(
                s["info"], a["y"], a["p"], NOISE, s["mean"], 1, 300, 1e-3, 10, 0, True,
                s["alpha"])["cache_handle"]
    return s


def _alpha(case, a, iterations):
    """(K + NOISE I)^-1 (y - mean) in 64 bits, rounded."""
    b = _dev64(a["y"]) - float(a["y"].mean())
    x = _solve64(case, _dev64(a["X"]), _dev64(a["p"]), b, iterations)
    return x.to(torch.float32).cpu().numpy()


# ---------------------------------------------------------------- the passes

def _fp(t):
    return C.cast(t.data_ptr(), C.POINTER(C.c_float))


def run(state):
    case, op = state["case"], state["case"]["op"]
    if op == "product":
        _lib.call("mgp_forward_matvec_device", state["provs"][0].handle, _fp(state["V"]),
                  case["t"], _fp(state["out"]))
        return state["out"]
    if op == "trace":
        return state["provs"][0].gradient_trace(state["L"], state["R"])
    if op == "lmc":
        out = np.empty_like(state["V"])
        _lib.call("mgp_lmc_forward_matvec", _lib.handles(state["provs"]), 2, case["tasks"],
                  _lib.fptr(state["A"]), _lib.fptr(state["noise"]), None, _lib.fptr(state["V"]),
                  case["t"], _lib.fptr(out))
        return out
    if op == "fit":
        gp = SingleOutputGP(_node(case))
        r = gp.fit(state["X"], state["y"], max_iterations=case["steps"], method="matrix_free")
        return {"params": r.params, "noise": float(r.noise), "mean": float(r.mean),
                "nll": np.asarray(r.nll_history)}
    if op == "serve":
        r = load_engine().predict_with_cache(state["info"], state["cache"], state["Xs"],
                                             state["p"], NOISE, state["mean"], 1)
        return {"mean": r["mean"], "variance": r["variance"]}
    r = load_engine().predict(state["info"], state["y"], state["Xs"], state["p"], NOISE,
                              state["mean"], 1, 300, 1e-3, 10, 0, True)
    return {"mean": r["mean"], "variance": r["variance"], "alpha": r["cached_alpha"]}


# ---------------------------------------------------------------- what a pass cannot do without

def work(case):
    op, n, d = case["op"], case["n"], case["d"]
    pair = lambda k, dims, cols: 3 * dims + VALUE_FLOPS[k] + 2 * cols  # noqa: E731
    half = n * (n + 1) / 2  # distinct kernel values of a square product
    if op == "product":
        t = case["t"]
        if case["dense"]:  # K is held: the values of one triangle, 4 bytes each
            return {"bytes": 4 * half + 8 * n * t, "flops": 2.0 * n * n * t}
        return {"bytes": 4 * n * (d + 2 * t),
                "flops": half * pair(case["kernel"], d, 0) + 2.0 * n * n * t}
    if op == "trace":
        t = case["t"]
        return {"bytes": 4 * n * (d + 2 * t),
                "flops": half * (pair(case["kernel"], d, 2 * t) + 2 * d + 4)}
    if op == "lmc":
        cols = case["t"] * case["tasks"]
        return {"bytes": 4 * n * (d + 2 * cols),
                "flops": half * (pair("rbf", d, 0) + pair("matern52", d, 0)) + 8.0 * n * n * cols}
    if op == "fit":  # at least 11 CG iterations of 11 columns and one trace a step
        one = half * pair(case["kernel"], d, 0) + 22.0 * n * n
        return {"bytes": case["steps"] * 11 * 4.0 * n * (d + 22),
                "flops": case["steps"] * (11 * one + half * (pair(case["kernel"], d, 22) + 2 * d))}
    rank = 200 if case["ard"] else 100
    cross = case["m"] * n * pair(case["kernel"], d, 1 + rank)
    if op == "serve":
        return {"bytes": 4.0 * n * (d + 1 + rank) + 4.0 * case["m"] * (d + 2), "flops": cross}
    solves = 0.5 * n * n * pair(case["kernel"], d, 0) + 2.0 * n * n
    return {"bytes": 4.0 * n * (d + 2 + rank) + 4.0 * n * rank * rank / 2,
            "flops": rank * solves + cross + 4.0 * n * rank * rank}


def tolerance(case):
    # about four times the largest error against 64 bits over 63 cases of these
    # ranges (3.7e-7 products, 2.0e-5 traces, 2.5e-5 the served mean, 1.1e-3
    # the mean of the first prediction, whose CG stops at 1e-3); a fit: the
    # path against itself with its sums in another order (1.2e-4)
    return {"rel": {"product": 2e-6, "lmc": 2e-6, "trace": 8e-5, "serve": 1e-4,
                    "predict": 5e-3, "fit": 5e-4}[case["op"]]}


def exact(case, seed):
    op = case["op"]
    if op == "fit":
        return None
    a = _inputs(case, seed)
    X = _dev64(a["X"])
    if op == "lmc":
        T, n, t = case["tasks"], case["n"], case["t"]
        V = _dev64(a["V"]).reshape(t * T, n)
        A, noise = _dev64(a["A"]), _dev64(a["noise"])
        out = noise[None, :, None] * V.reshape(t, T, n)
        for s, kernel in enumerate(("rbf", "matern52")):
            one = {"kernel": kernel, "ard": False}
            KV = _matvec64(one, X, X, _dev64(a["p"][s]), V).reshape(t, T, n)
            out += torch.einsum("ij,cjn->cin", A[s], KV)
        return out.reshape(t, T * n).cpu().numpy()
    p = _dev64(a["p"])
    if op == "product":
        V = _dev64(a["V"])
        return _matvec64(case, X, X, p, V) + NOISE * V
    if op == "trace":
        L, R = _dev64(a["L"]), _dev64(a["R"])
        p.requires_grad_(True)
        step = max(16, (1 << 23) // case["n"])
        for i in range(0, case["n"], step):
            W = L[:, i:i + step].T @ R
            (W * _block(case, X[i:i + step], X, p)).sum().backward()
        return p.grad.cpu().numpy()
    alpha = (_dev64(a["y"]) - float(a["y"].mean()))
    alpha = (_dev64(_alpha(case, a, 100)) if op == "serve"
             else _solve64(case, X, p, alpha, 300))
    mean = _matvec64(case, _dev64(a["Xs"]), X, p, alpha[None])[0] + float(a["y"].mean())
    out = {"mean": mean.cpu().numpy(), "variance": None}
    if op == "predict":
        out["alpha"] = None
    return out
