"""Density-only K of densities that its Cholesky factor gives up early, against the CPU oracle: a small tail behind
the occupied space (from 1e-3 and from 1e-7 of it, both sides of the limit of 1e-4 of the largest diagonal) and
a slowly falling spectrum (found out after eight columns), in the one-work-group kernel on both sides of the size
from which it extrapolates (nbf 158 / 160) and in the one of a launch a column (nbf 257); one and two spins.
Bound 1e-11, as tests/test_gpu_dm_factor.py."""
import numpy as np
import pytest

from oracle import oracle as orc
from rest_amd import jk

pytestmark = pytest.mark.gpu


def density(kind, n, rng):
    q = np.linalg.qr(rng.standard_normal((n, n)))[0]
    o = n // 5
    lam = {"tail 1e-3": 2.0 * (np.arange(n) < o) + 1e-3 * 10.0 ** -np.linspace(0, 12, n),
           "tail 1e-7": 2.0 * (np.arange(n) < o) + 1e-7 * 10.0 ** -np.linspace(0, 8, n),
           "graded": np.linspace(1.0, 0.1, n), "low": 2.0 * (np.arange(n) < o)}[kind]
    d = (q * lam) @ q.T
    return 0.5 * (d + d.T)


@pytest.mark.parametrize("n", [30, 158, 160, 256, 257])
@pytest.mark.parametrize("kinds", [("tail 1e-3",), ("tail 1e-7", "low"), ("graded",), ("low", "graded")])
def test_densities_given_up(n, kinds):
    print(f"[gpu-case] density-only K nbf={n} {kinds}", flush=True)
    rng = np.random.default_rng(n + len(kinds))
    b = rng.standard_normal((n * (n + 1) // 2, 6)) / np.sqrt(6)
    ds = [density(k, n, rng) for k in kinds]
    ref = orc.vk_upper_dm(b, True, ds, len(ds), -0.5)
    with jk.DeviceRI(n, 6) as ri:
        ri.set_rimatr(b)
        assert np.abs(ri.vk_dm(ds, len(ds), -0.5) - ref).max() <= 1e-11
