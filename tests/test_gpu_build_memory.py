"""What a B build leaves on its context: within the workspace limit its scratch stays for the next build, beyond
the limit all of it is given back, on the route of the polar factor and on that of the eigenpairs (a threshold of
half the smallest eigenvalue keeps every eigenvalue but is above the polar route's bound).  B is the same either
way, bit for bit.  Eight waters: metric matrices of 6.5 MB, a slab of integrals of 134 MB."""
import numpy as np
import pytest

from rest_amd import jk, ri
from rest_amd import workload as wl

pytestmark = pytest.mark.gpu


def built(m, thr, limit):
    """(device bytes held by a context after its build, B)"""
    free = jk.device_memory()[0]
    with jk.DeviceRI(m.nbf, m.naux) as r:
        if limit:
            r.set_workspace_limit(limit)
        m.build_rimatr(r, threshold=thr)
        return free - jk.device_memory()[0], r.get_rimatr()


def test_build_gives_back_what_exceeds_the_limit():
    m = ri.Molecule.water_cluster(wl.water_cluster(4, 8))
    lam0 = np.linalg.eigvalsh(m.int2c2e())[0]
    slab = m.nbf * (m.nbf + 1) // 2 * m.naux * 8
    built(m, 1e-8, 0)                                   # libraries and code objects loaded
    for thr in (1e-8, 0.5 * lam0):
        print(f"[gpu-case] build memory, {m.naux} auxiliary functions, threshold {thr:.1e}", flush=True)
        kept, b0 = built(m, thr, 0)
        given, b1 = built(m, thr, 1 << 20)
        print(f"held {kept} within the limit, {given} beyond it", flush=True)
        assert np.array_equal(b0, b1)
        assert kept - given >= slab


def test_build_between_exchange_builds():
    """A K call before the build leaves a workspace that the build may use, whatever the limit, and B does not
    depend on it."""
    m = ri.Molecule.water_cluster(wl.water_cluster(4, 3))
    ref = built(m, 1e-8, 0)[1]
    c = np.linalg.qr(np.random.default_rng(1).standard_normal((m.nbf, m.nbf)))[0]
    with jk.DeviceRI(m.nbf, m.naux) as r:
        r.set_workspace_limit(1 << 20)
        for _ in range(2):
            m.build_rimatr(r)
            assert np.array_equal(r.get_rimatr(), ref)
            r.set_workspace_limit(0)
            r.vk_occ([c], [m.nbf - 1], [np.ones(m.nbf)], 1)
            r.set_workspace_limit(1 << 20)
