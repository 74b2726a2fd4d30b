"""Stochastic Lanczos quadrature on the host: first eigenvector components alone.

``slq_logdet`` keeps one row of the eigenvector matrix; it must be the row the
full decomposition gives, bit for bit, and the estimate that of numpy's eigh.
"""
import subprocess
from pathlib import Path

import numpy as np
import pytest

CSRC = Path(__file__).resolve().parent.parent / "mojogp_amd" / "csrc"

MAIN = r"""
#include "host_numerics.h"
#include <cstdio>
#include <cstring>
int main(int, char**) {
  int probes, m;
  long n;
  if (std::scanf("%d %d %ld", &probes, &m, &n) != 3) return 2;
  std::vector<std::vector<float>> d(probes, std::vector<float>(m)), e(probes);
  for (int p = 0; p < probes; ++p) {
    for (auto& v : d[p]) if (std::scanf("%f", &v) != 1) return 2;
    e[p].resize(m > 0 ? m - 1 : 0);
    for (auto& v : e[p]) if (std::scanf("%f", &v) != 1) return 2;
    std::vector<double> dd(d[p].begin(), d[p].end()), ee(e[p].begin(), e[p].end()), a, b, V, f;
    const bool ok = mgp::tridiag_eigh(dd, ee, a, &V), ok1 = mgp::tridiag_eigh(dd, ee, b, &f, 1);
    if (ok != ok1 || a != b || f.size() != (size_t)m) return 3;
    if (m && std::memcmp(V.data(), f.data(), m * sizeof(double))) return 4;
  }
  std::printf("%.9g\n", mgp::slq_logdet(d, e, n));
}
"""


@pytest.fixture(scope="module")
def exe(tmp_path_factory):
    tmp = tmp_path_factory.mktemp("slq")
    (tmp / "main.cpp").write_text(MAIN)
    out = tmp / "slq"
    subprocess.run(["g++", "-std=c++17", "-O2", f"-I{CSRC}", "-x", "c++", str(tmp / "main.cpp"),
                    str(CSRC / "host_numerics.hip"), "-o", str(out)], check=True)
    return out


@pytest.mark.parametrize("m", [1, 2, 3, 30, 50])
def test_first_components(exe, m):
    rng = np.random.default_rng(m)
    probes, n = 5, 1000
    diag = (2.0 + rng.random((probes, m))).astype(np.float32)
    off = (0.9 * rng.random((probes, max(m - 1, 0)))).astype(np.float32)
    if m > 2:
        off[0, 1] = 0.0  # a split matrix
    text = f"{probes} {m} {n}\n" + "\n".join(
        " ".join(f"{v:.9g}" for v in np.concatenate([diag[p], off[p]])) for p in range(probes))
    got = float(subprocess.run([str(exe)], input=text, text=True, check=True,
                               capture_output=True, timeout=60).stdout)
    ref = 0.0
    for p in range(probes):
        T = np.diag(diag[p].astype(np.float64))
        T += np.diag(off[p].astype(np.float64), 1) + np.diag(off[p].astype(np.float64), -1)
        lam, V = np.linalg.eigh(T)
        ref += float(np.sum(V[0] ** 2 * np.log(lam))) / probes
    # m fp32 terms and their sum: under (m + 4) 2^-24 of sum |terms|
    assert abs(got - n * ref) <= (m + 4) * 2.0 ** -23 * n * max(abs(ref), 1.5)
