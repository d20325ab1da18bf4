"""The eigensolver of the SCF at the edges of its sizes: 40 / 41 (rocSOLVER below), 64 / 65, 128 / 129 (register
blocks), 192 / 193 (a launch a column above), 320 / 321, 512 / 513, 1024 / 1025 (rocSOLVER above); and spectra with clusters: gaps of 1e-7 (orthogonalised), exact
fourfold degeneracy (divide and conquer on the same tridiagonal).  With B = 0 the Fock matrix of a guess
step is H, so its orbitals solve H C = S C eps.  Bounds: an eigensolver's backward error of n eps |F'|,
with F' = S^(-1/2) H S^(-1/2) and S within a factor 3 of one: 10 n eps |H| on H C - S C eps and 10 n eps on
C^T S C - 1."""
import numpy as np
import pytest
import scipy.linalg

from rest_amd import jk
from rest_amd import scf as rs

pytestmark = pytest.mark.gpu


def spectrum(kind, n, rng):
    if kind == "random":
        return None
    step = {"close": 1e-7, "fourfold": 0.0}[kind]
    return np.repeat(np.linspace(-20.0, 5.0, (n + 3) // 4), 4)[:n] + step * (np.arange(n) % 4)


@pytest.mark.parametrize("n,kind", [(40, "random"), (41, "random"), (64, "random"), (65, "random"), (96, "close"),
                                    (128, "random"), (129, "fourfold"), (191, "close"), (192, "random"),
                                    (192, "fourfold"), (193, "random"), (256, "close"), (320, "random"), (321, "fourfold"),
                                    (512, "random"), (513, "close"), (1024, "random"), (1025, "random")])
def test_guess_step_eigenpairs(n, kind):
    print(f"[gpu-case] eigenpairs n={n} {kind}", flush=True)
    rng = np.random.default_rng(n)
    a = rng.standard_normal((n, n))
    if kind == "random":
        S = np.eye(n) + 0.1 * (a + a.T) / np.sqrt(n)
        b = rng.standard_normal((n, n))
        H = (b + b.T) / 2
    else:
        S = np.eye(n)
        q = np.linalg.qr(a)[0]
        H = (q * spectrum(kind, n, rng)) @ q.T
        H = (H + H.T) / 2
    with jk.DeviceRI(n, 1) as r:
        r.set_rimatr(np.zeros((n * (n + 1) // 2, 1)))
        c = rs.guess_step(r, S, H, 0.0, (2 * (n // 4),), np.zeros((n, n)))[2]
    C = np.asarray(c).reshape(n, n)
    eps = np.diag(C.T @ H @ C)
    ref = scipy.linalg.eigh(H, S, eigvals_only=True)
    tol = 10 * n * 2.3e-16
    hn = np.abs(ref).max()
    assert np.abs(C.T @ S @ C - np.eye(n)).max() <= tol
    assert np.abs(H @ C - S @ C * eps).max() <= tol * hn
    assert np.abs(eps - ref).max() <= tol * hn
