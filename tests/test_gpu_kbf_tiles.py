"""GPU parity of the BF16 K tiles at the sizes where their shape changes: nbf around a 32-deep MFMA step,
the 128-row tiles and the step from four to eight waves (512); column counts around the 32-column runs
and the widest half-transform tile (192 columns); odd run counts (a k-block half empty); one and two
spins, one of them signed; several auxiliary chunks.  Against the float64 oracle.  Three planes: 2e-6 of
the largest element (as tests/test_gpu_kbf.py).  Two planes: a product keeps 2^-16 of its operands'
magnitudes in each of two stages, at most 2 x 3 x 2^-16 < 2e-4 of the largest (a diagonal
element, a sum of squares); a plane product left out costs 2^-8."""
import numpy as np
import pytest

from oracle import oracle as orc
from rest_amd import jk

pytestmark = pytest.mark.gpu
STORE = jk.STORE_FP64 | jk.STORE_FP32 | jk.STORE_BF16


@pytest.mark.parametrize("nbf,naux,nw,ns", [
    (31, 5, (1, 1), 1), (33, 11, (31, 33), 2), (127, 9, (64, 1), 1), (129, 3, (65, 30), 2), (193, 13, (97, 96), 1),
    (256, 6, (160, 3), 2), (257, 7, (193, 1), 1), (512, 2, (161, 31), 1), (513, 3, (129, 70), 2),
])
def test_bf16_tile_edges(nbf, naux, nw, ns):
    print(f"[gpu-case] BF16 K tiles nbf={nbf} naux={naux} nw={nw} ns={ns}", flush=True)
    rng = np.random.default_rng(nbf * 11 + naux)
    npair = nbf * (nbf + 1) // 2
    b = rng.standard_normal((npair, naux)) / np.sqrt(naux)
    nstate = max(nw)
    cs = [rng.standard_normal((nbf, nstate)) / np.sqrt(nbf) for _ in range(ns)]
    occs = [rng.uniform(0.2, 2.0, nstate) for _ in range(ns)]
    if nw[-1] > 1:
        occs[-1][0] = -0.3
    homo = [nw[s] - 1 for s in range(ns)]
    ref = orc.vk_upper_occ(b, True, cs, homo, occs, ns, -0.5)
    big = np.abs(ref).max()
    with jk.DeviceRI(nbf, naux) as ri:
        ri.set_rimatr(b, STORE)
        x2 = ri.vk_occ(cs, homo, occs, ns, -0.5, prec=jk.PREC_BF16X2)
        x3 = ri.vk_occ(cs, homo, occs, ns, -0.5, prec=jk.PREC_BF16X3)
        ri.set_workspace_limit(6 << 20)
        many = ri.vk_occ(cs, homo, occs, ns, -0.5, prec=jk.PREC_BF16X3)
    assert np.abs(x3 - ref).max() <= 2e-6 * big and np.abs(many - ref).max() <= 2e-6 * big
    assert np.abs(x2 - ref).max() <= 2e-4 * big
