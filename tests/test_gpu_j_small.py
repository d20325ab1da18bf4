"""J on both sides of its two-launch route (2048 packed pairs, 1024 auxiliary functions) and at its smallest, one
and two spins, upper-triangle and full densities, FP64 and FP32 B; also the splits of the larger route.
Against the CPU oracle: FP64 1e-12 n of the largest element (sums of naux and npair products), FP32 B 1e-6
of it (B's own rounding, FP64 sums)."""
import numpy as np
import pytest

from oracle import oracle as orc
from rest_amd import jk

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nbf,naux,ns", [
    (1, 1, 1), (2, 7, 2), (5, 8, 1), (24, 113, 2), (62, 17, 1), (63, 1024, 1), (63, 1025, 2), (64, 1024, 1),
    (65, 33, 2), (100, 700, 1),
])
def test_j_small_edges(nbf, naux, ns):
    print(f"[gpu-case] J nbf={nbf} naux={naux} ns={ns}", flush=True)
    rng = np.random.default_rng(nbf * 13 + naux)
    npair = nbf * (nbf + 1) // 2
    b = rng.standard_normal((npair, naux)) / np.sqrt(naux)
    ds = [rng.standard_normal((nbf, nbf)) for _ in range(ns)]       # not symmetric: the upper triangle counts
    up = orc.vj_upper_rimatr(b, ds, ns, 0.7)
    b3 = np.zeros((nbf, nbf, naux))
    for j in range(nbf):
        for i in range(j + 1):
            b3[i, j] = b3[j, i] = b[j * (j + 1) // 2 + i]
    full = orc.vj_upper_ri3fn(b3, ds, ns, 0.7)
    big = max(np.abs(up).max(), np.abs(full).max())
    with jk.DeviceRI(nbf, naux) as ri:
        ri.set_rimatr(b, jk.STORE_FP64 | jk.STORE_FP32)
        for _ in range(2):
            assert np.abs(ri.vj(ds, ns, 0.7) - up).max() <= 1e-12 * nbf * big
        assert np.abs(ri.vj(ds, ns, 0.7, full_dm=True) - full).max() <= 1e-12 * nbf * big
        assert np.abs(ri.vj(ds, ns, 0.7, prec=jk.PREC_FP32) - up).max() <= 1e-6 * nbf * big


@pytest.mark.parametrize("nbf", [24, 181, 182])
def test_host_calls_on_both_sides_of_the_pinned_size(nbf):
    """Densities of 181 x 181 pass through 256 KiB of pinned memory, of 182 x 182 directly; J, both K routes and two
    contexts in turn must each return their own results."""
    rng = np.random.default_rng(nbf)
    naux, nocc = 19, 5
    npair = nbf * (nbf + 1) // 2
    b = [rng.standard_normal((npair, naux)) / np.sqrt(naux) for _ in range(2)]
    with jk.DeviceRI(nbf, naux) as r0, jk.DeviceRI(nbf, naux) as r1:
        for r, x in zip((r0, r1), b):
            r.set_rimatr(x)
        for it in range(3):
            for r, x in zip((r0, r1), b):
                c = rng.standard_normal((nbf, nocc)) / np.sqrt(nbf)
                occ = rng.uniform(0.5, 2.0, nocc)
                d = (c * occ) @ c.T
                j, k = orc.vj_upper_rimatr(x, [d], 1, 1.0), orc.vk_upper_occ(x, True, [c], [nocc - 1], [occ], 1, -0.5)
                big = max(np.abs(j).max(), np.abs(k).max())
                assert np.abs(r.vj([d], 1) - j).max() <= 1e-12 * nbf * big
                assert np.abs(r.vk_occ([c], [nocc - 1], [occ], 1, -0.5) - k).max() <= 1e-12 * nbf * big
                assert np.abs(r.vk_dm([d], 1, -0.5) - k).max() <= 1e-12 * nbf * big
