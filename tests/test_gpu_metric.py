"""V^(-1/2) of the metric at the edges of its two routes: sizes around the 64-pivot blocks, and thresholds on
either side of the smallest eigenvalue (all eigenvalues kept: the polar factor; fewer: the eigenpairs).
Both must give B B^T = X V^+ X^T over the kept space: compared through B V^(1/2) = X P with numpy's
eigenpairs of the host metric, to 1e-9 of the largest integral (n eps |V| / lambda_min, as
tests/test_gpu_build.py), and the kept count with numpy's."""
import numpy as np
import pytest

from rest_amd import jk, ri
from rest_amd import workload as wl

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("waters,cut", [(1, 0.5), (1, 2.0), (2, 0.1), (2, 3.0), (4, 0.1), (4, 2.0), (5, 0.0)])
def test_both_metric_routes(waters, cut):
    m = ri.Molecule.water_cluster(wl.water_cluster(3, waters))
    V = m.int2c2e()
    lam, U = np.linalg.eigh(V)
    thr = cut * lam[0]
    print(f"[gpu-case] metric {waters} waters, naux {m.naux}, threshold {thr:.2e}", flush=True)
    keep = lam > thr
    root = (U[:, keep] * np.sqrt(lam[keep])) @ U[:, keep].T
    proj = U[:, keep] @ U[:, keep].T
    X = m.int3c2e_packed()
    with jk.DeviceRI(m.nbf, m.naux) as r:
        info = m.build_rimatr(r, threshold=thr)
        B = r.get_rimatr()
    assert info["naux_kept"] == int(keep.sum())
    assert np.abs(B @ root - X @ proj).max() <= 1e-9 * np.abs(X).max()


def test_metric_beyond_one_work_group():
    """More than 2048 auxiliary functions (a launch a pivot).  A threshold of half the smallest eigenvalue keeps
    every eigenvalue but is above the bound 1/|V^(-1/2)|^2, so it takes the eigenpairs: both routes must give
    the same B, compared through J of a random density to 1e-9 (as above)."""
    m = ri.Molecule.water_cluster(wl.water_cluster(5, 19))
    assert m.naux > 2048
    lam0 = np.linalg.eigvalsh(m.int2c2e())[0]
    print(f"[gpu-case] metric of {m.naux} functions, smallest eigenvalue {lam0:.2e}", flush=True)
    rng = np.random.default_rng(1)
    d = rng.standard_normal((m.nbf, m.nbf))
    d = d + d.T
    out = []
    for thr in (1e-8, 0.5 * lam0):
        with jk.DeviceRI(m.nbf, m.naux) as r:
            assert m.build_rimatr(r, threshold=thr)["naux_kept"] == m.naux
            out.append(r.vj([d], 1)[0])
    assert np.abs(out[0] - out[1]).max() <= 1e-9 * np.abs(out[1]).max()
