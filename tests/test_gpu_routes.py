"""Which solver ran: every fast route has a fallback that gives the same numbers, so each is asserted by the
context's route counts.  Density-only K: which densities take the Cholesky factor, the eigenpairs, the general
route, at the edges of its kernels.  SCF eigenproblems: spectra that the own kernels must solve, equal
eigenvalues that they must hand on, sizes outside them.  Metric: the polar factor with every eigenvalue kept,
the eigenpairs for a threshold above its bound 1 / |V^(-1/2)|^2 on the smallest eigenvalue, and with more than 1024 functions (each thread of the pivot panel then
owns two rows) its B against the integrals, B V^(1/2) = X to 1e-9 as tests/test_gpu_metric.py."""
import numpy as np
import pytest

from rest_amd import jk, ri
from rest_amd import scf as rs
from rest_amd import workload as wl

pytestmark = pytest.mark.gpu


def taken(r):
    return {k: v for k, v in r.route_counts().items() if v}


def density(kind, n, rng):
    if kind == "zero":
        return np.zeros((n, n))
    if kind == "general":
        return rng.standard_normal((n, n))
    if kind == "swap":
        d = np.zeros((n, n))
        d[0, n - 1] = d[n - 1, 0] = 0.3
        return d
    q = np.linalg.qr(rng.standard_normal((n, n)))[0]
    o = n // 5
    lam = {"one": np.arange(n) < 1, "occ": 2.0 * (np.arange(n) < o), "mixed occ": np.where(np.arange(n) < o, rng.uniform(0.5, 2, n), 0),
           "most": 1.0 * (np.arange(n) < (n // 2 if n <= 256 else n // 4 + 64)), "full": np.ones(n), "graded": np.linspace(1, 0.1, n),
           "tail": 2.0 * (np.arange(n) < o) + 1e-6, "negative": -1.0 * (np.arange(n) < o)}[kind]
    d = (q * lam) @ q.T
    return 0.5 * (d + d.T)


@pytest.mark.parametrize("n", [20, 111, 112, 256, 257])
@pytest.mark.parametrize("kinds,route", [
    (("zero",), "cholesky"), (("one",), "cholesky"), (("occ",), "cholesky"), (("mixed occ", "occ"), "cholesky"),
    (("most",), "cholesky"), (("full",), "eigenpairs"), (("graded",), "eigenpairs"), (("tail",), "eigenpairs"),
    (("swap",), "eigenpairs"), (("occ", "negative"), "eigenpairs"), (("occ", "general"), "general")])
def test_density_routes(n, kinds, route):
    print(f"[gpu-case] route of the density-only K nbf={n} {kinds}", flush=True)
    rng = np.random.default_rng(n)
    ds = [density(k, n, rng) for k in kinds]
    with jk.DeviceRI(n, 3) as r:
        r.fill_synthetic(1, jk.STORE_FP64 | jk.STORE_FP32)
        r.vk_dm(ds, len(ds), 1.0)
        assert taken(r) == {"dm_" + route: 1}
        if route == "cholesky":
            r.vk_dm(ds, len(ds), 1.0, prec=jk.PREC_FP32)   # the lower precisions keep the eigenpairs
            assert taken(r) == {"dm_cholesky": 1, "dm_eigenpairs": 1}


@pytest.mark.parametrize("n", [41, 64, 65, 128, 129, 192, 193, 320, 321, 512, 513, 1024])
@pytest.mark.parametrize("kind,own", [("random", 2), ("close", 1), ("fourfold", 0)])
def test_eigen_routes(n, kind, own):
    """A guess step solves S and F.  S is the identity for the two made spectra: equal eigenvalues, handed on."""
    print(f"[gpu-case] route of the eigenproblem n={n} {kind}", flush=True)
    rng = np.random.default_rng(n)
    a, b = rng.standard_normal((2, n, n))
    S, H = np.eye(n), (b + b.T) / 2
    if kind == "random":
        S = S + 0.1 * (a + a.T) / np.sqrt(n)
    else:
        lam = np.repeat(np.linspace(-20.0, 5.0, (n + 3) // 4), 4)[:n] + (1e-7 if kind == "close" else 0.0) * (np.arange(n) % 4)
        q = np.linalg.qr(a)[0]
        H = (q * lam) @ q.T
        H = (H + H.T) / 2
    with jk.DeviceRI(n, 1) as r:
        r.set_rimatr(np.zeros((n * (n + 1) // 2, 1)))
        rs.guess_step(r, S, H, 0.0, (2 * (n // 4),), np.zeros((n, n)))
        got = taken(r)
    assert got.get("eig_own", 0) == own and got.get("eig_divide", 0) == 2 - own and "eig_rocsolver" not in got


@pytest.mark.parametrize("n", [40, 1025])
def test_sizes_left_to_rocsolver(n):
    print(f"[gpu-case] eigenproblem n={n}", flush=True)
    b = np.random.default_rng(n).standard_normal((n, n))
    with jk.DeviceRI(n, 1) as r:
        r.set_rimatr(np.zeros((n * (n + 1) // 2, 1)))
        rs.guess_step(r, np.eye(n), (b + b.T) / 2, 0.0, (2 * (n // 4),), np.zeros((n, n)))
        got = taken(r)
    assert got["eig_rocsolver"] == 2 and "eig_own" not in got and "eig_divide" not in got


@pytest.mark.parametrize("waters", [1, 5, 10, 19])
def test_metric_routes(waters):
    m = ri.Molecule.water_cluster(wl.water_cluster(3, waters))
    V = m.int2c2e()
    lam, U = np.linalg.eigh(V)
    print(f"[gpu-case] metric route, {m.naux} functions", flush=True)
    with jk.DeviceRI(m.nbf, m.naux) as r:
        m.build_rimatr(r, threshold=1e-8)
        assert taken(r) == {"metric_polar": 1}
        if waters == 10:
            X = m.int3c2e_packed()
            assert np.abs(r.get_rimatr() @ ((U * np.sqrt(lam)) @ U.T) - X).max() <= 1e-9 * np.abs(X).max()
        polar = 1
        for share in (0.5, 0.999):
            m.build_rimatr(r, threshold=share * lam[0])
            polar += 1.0 / (1.0 / lam).sum() > share * lam[0]
        assert taken(r) == {"metric_polar": polar, "metric_eigenpairs": 3 - polar} and polar < 3


@pytest.mark.parametrize("waters,share", [(1, 0.1), (2, 0.5), (5, 0.02), (19, 0.3)])
def test_threshold_among_the_eigenvalues(waters, share):
    """A threshold above that share of the eigenvalues ends the factor at a pivot below it: the eigenpairs, and as
    many of them as numpy keeps; B V^(1/2) = X P over the kept space to 1e-9."""
    m = ri.Molecule.water_cluster(wl.water_cluster(3, waters))
    lam, U = np.linalg.eigh(m.int2c2e())
    cut = int(share * m.naux)
    thr = float(np.sqrt(lam[cut - 1] * lam[cut]))
    print(f"[gpu-case] metric of {m.naux} functions, threshold {thr:.2e} above {cut} eigenvalues", flush=True)
    with jk.DeviceRI(m.nbf, m.naux) as r:
        assert m.build_rimatr(r, threshold=thr)["naux_kept"] == m.naux - cut
        assert taken(r) == {"metric_eigenpairs": 1}
        if waters < 10:
            X = m.int3c2e_packed()
            kept = U[:, cut:]
            d = r.get_rimatr() @ (kept * np.sqrt(lam[cut:])) @ kept.T - X @ kept @ kept.T
            assert np.abs(d).max() <= 1e-9 * np.abs(X).max()
