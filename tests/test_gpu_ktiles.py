"""GPU parity of the K tiles at the sizes where their choice changes: nbf at the edges of the 64- and
128-row tiles and of a 16-function k-block, column counts that take each tile width, negative and empty
occupations, one and two spins, several auxiliary chunks; against the CPU oracle.  FP64: max-abs 1e-11.
FP32: 2e-5 of the largest element (sums of at most 4096 FP32 products, as tests/test_gpu_jk.py states)."""
import numpy as np
import pytest

from oracle import oracle as orc
from rest_amd import jk

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nbf,naux,nw,ns", [
    (15, 9, (3, 1), 1), (63, 17, (16, 15), 2), (64, 11, (33, 2), 1), (65, 40, (17, 40), 2),
    (127, 13, (65, 1), 1), (128, 21, (96, 16), 1), (129, 8, (97, 81), 2), (144, 19, (112, 3), 1),
    (193, 33, (81, 79), 2), (257, 9, (129, 7), 1),
])
def test_tile_edges(nbf, naux, nw, ns):
    print(f"[gpu-case] K tiles nbf={nbf} naux={naux} nw={nw} ns={ns}", flush=True)
    rng = np.random.default_rng(nbf * 7 + naux)
    npair = nbf * (nbf + 1) // 2
    b = rng.standard_normal((npair, naux)) / np.sqrt(naux)
    nstate = max(nw)
    cs = [rng.standard_normal((nbf, nstate)) / np.sqrt(nbf) for _ in range(ns)]
    occs = [rng.uniform(0.2, 2.0, nstate) for _ in range(ns)]
    occs[-1][0] = -0.7           # one spin signed, the other not
    if nw[-1] > 2:
        occs[-1][2] = 0.0
    homo = [nw[s] - 1 for s in range(ns)]
    ref = orc.vk_upper_occ(b, True, cs, homo, occs, ns, -0.5)
    big = np.abs(ref).max()
    with jk.DeviceRI(nbf, naux) as ri:
        ri.set_rimatr(b, jk.STORE_FP64 | jk.STORE_FP32)
        one = ri.vk_occ(cs, homo, occs, ns, -0.5)
        f32 = ri.vk_occ(cs, homo, occs, ns, -0.5, prec=jk.PREC_FP32)
        ri.set_workspace_limit(3 << 20)
        many = ri.vk_occ(cs, homo, occs, ns, -0.5)
    assert np.abs(one - ref).max() <= 1e-11 and np.abs(many - ref).max() <= 1e-11
    assert np.abs(f32 - ref).max() <= 2e-5 * big
