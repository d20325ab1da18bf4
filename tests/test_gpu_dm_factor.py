"""The density-only K's choice of columns against the CPU oracle: Cholesky factor of a low-rank density at the
edges of its kernels (256 functions, its column limits), and the densities it must leave to the
eigenpairs (indefinite with a zero diagonal, negative, rank above the limit), one and two spins.
Bound: 1e-11, as tests/test_gpu_jk.py (the columns reproduce D to 1e-13 of its largest element)."""
import numpy as np
import pytest

from oracle import oracle as orc
from rest_amd import jk

pytestmark = pytest.mark.gpu


def density(kind, n, rng):
    if kind == "zero":
        return np.zeros((n, n))
    if kind == "swap":                     # symmetric, zero diagonal, indefinite
        d = np.zeros((n, n))
        d[0, n - 1] = d[n - 1, 0] = 0.3
        return d
    q = np.linalg.qr(rng.standard_normal((n, n)))[0]
    r = {"one": 1, "occ": max(1, n // 5), "half": max(1, n // 2), "over": min(n, n // 2 + 1), "full": n, "neg": n // 3 + 1}[kind]
    lam = rng.uniform(0.5, 2.0, r) * (-1.0 if kind == "neg" else 1.0)
    d = (q[:, :r] * lam) @ q[:, :r].T
    return 0.5 * (d + d.T)


@pytest.mark.parametrize("n,naux", [(2, 5), (33, 12), (200, 7), (256, 5), (257, 5)])
@pytest.mark.parametrize("kinds", [("occ",), ("one", "zero"), ("half", "occ"), ("over",), ("swap",), ("neg", "occ"),
                                   ("full",)])
def test_density_columns(n, naux, kinds):
    print(f"[gpu-case] density-only K nbf={n} {kinds}", flush=True)
    rng = np.random.default_rng(n + len(kinds))
    b = rng.standard_normal((n * (n + 1) // 2, naux)) / np.sqrt(naux)
    ds = [density(k, n, rng) for k in kinds]
    ref = orc.vk_upper_dm(b, True, ds, len(ds), -0.5)
    with jk.DeviceRI(n, naux) as ri:
        ri.set_rimatr(b)
        assert np.abs(ri.vk_dm(ds, len(ds), -0.5) - ref).max() <= 1e-11
