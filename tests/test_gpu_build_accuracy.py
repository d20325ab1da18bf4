"""B against X V^(-1/2) with the root formed in 80 bits from the host's integrals.  V is ill-conditioned: rounding its
elements to 64 bits (3e-16 of it, whichever engine computes them) already moves B by 0.8e-12 to 1.2e-12 of its norm
for one to three waters, measured against integrals in 80 bits, and the device's V is rounded apart
from the host's: 2 x 1.2e-12, doubled for the products' own rounding and B's largest element, 5e-12."""
import numpy as np
import pytest

from rest_amd import jk, ri
from rest_amd import workload as wl

pytestmark = pytest.mark.gpu


def inverse_root(V):
    """V^(-1/2) in extended precision: coupled Newton-Schulz steps, the cubic closest to one on [l, 1] while l is small."""
    V = V.astype(np.longdouble)
    one = np.eye(len(V), dtype=np.longdouble)
    norm = np.abs(V).sum(1).max()
    Y, Z, l = V / norm, one, np.sqrt(np.longdouble(1e-7) / norm)
    for _ in range(80):
        W = Z @ Y
        if np.abs(W - one).max() < 1e-12:
            break
        a, b = np.longdouble(1.5), np.longdouble(0.5)
        if l < 0.9:
            q = 1 + l + l * l
            m = 2 * q * np.sqrt(q / 3) / 3
            a, b, l = q / m, 1 / m, (q - 1) / m
        T = a * one - b * W
        Y, Z = Y @ T, T @ Z
    return (Z / np.sqrt(norm)).astype(float)


@pytest.mark.parametrize("waters,seed", [(1, 1), (1, 2), (1, 8), (2, 1), (2, 3)])
def test_b_against_extended_precision(waters, seed):
    m = ri.Molecule.water_cluster(wl.water_cluster(seed, waters))
    V = m.int2c2e()
    ref = m.int3c2e_packed() @ inverse_root(0.5 * (V + V.T))
    with jk.DeviceRI(m.nbf, m.naux) as r:
        m.build_rimatr(r)
        B = r.get_rimatr()
    err = np.linalg.norm(B - ref) / np.linalg.norm(ref), np.abs(B - ref).max() / np.abs(ref).max()
    print(f"[gpu-case] B of {m.naux} functions: {err[0]:.1e} of its norm, {err[1]:.1e} of its largest element", flush=True)
    assert max(err) <= 5e-12
