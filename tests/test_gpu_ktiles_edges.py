"""GPU parity of the FP64 / FP32 K tiles where tests/test_gpu_ktiles.py does not go: the single-problem FP64 SYRK of
128-row tiles at functions that do not fill them, two spins, signed columns, one and several chunks; and the batch's
tiles: both row classes of the half-transform by the cut of the configuration, every column group and its
remainders, both classes of the SYRK (64 rows, 128 beyond 640 functions at FP64) in one batch, negative and empty
weights, fewer auxiliary columns than XCDs.  Against the CPU oracle.  FP64: max-abs 1e-11; FP32: K 2e-5 of the largest
element (sums of at most 4096 FP32 products), J 1e-6 of it (B held in FP32, FP64 sums), as the tests beside."""
import numpy as np
import pytest

from oracle import oracle as orc
from rest_amd import jk

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nbf,naux,nw,ns", [(700, 9, (33, 17), 2), (740, 13, (7, 2), 1), (1000, 6, (48, 65), 2)])
def test_syrk_of_128_row_tiles(nbf, naux, nw, ns):
    print(f"[gpu-case] 128-row K tiles nbf={nbf} naux={naux} nw={nw} ns={ns}", flush=True)
    rng = np.random.default_rng(nbf)
    b = rng.standard_normal((nbf * (nbf + 1) // 2, naux)) / np.sqrt(naux)
    nstate = max(nw)
    cs = [rng.standard_normal((nbf, nstate)) / np.sqrt(nbf) for _ in range(ns)]
    occs = [rng.uniform(0.2, 2.0, nstate) for _ in range(ns)]
    occs[-1][1] = -0.7
    homo = [nw[s] - 1 for s in range(ns)]
    ref = orc.vk_upper_occ(b, True, cs, homo, occs, ns, -0.5)
    with jk.DeviceRI(nbf, naux) as r:
        r.set_rimatr(b)
        one = r.vk_occ(cs, homo, occs, ns, -0.5)
        r.set_workspace_limit(32 << 20)
        many = r.vk_occ(cs, homo, occs, ns, -0.5)
    assert np.abs(one - ref).max() <= 1e-11 and np.abs(many - ref).max() <= 1e-11


@pytest.mark.parametrize("prec", ["fp64", "fp32"])
@pytest.mark.parametrize("cut", [0, 1 << 30])
@pytest.mark.parametrize("shapes", [
    [(1, 1, 1), (16, 9, 4), (33, 7, 32), (63, 3, 33), (64, 8, 64)],
    [(65, 10, 65), (96, 5, 80), (127, 9, 81), (128, 17, 96), (129, 8, 97)],
    [(191, 6, 128), (192, 4, 129), (257, 3, 160), (200, 5, 161)],
    [(640, 5, 17), (641, 9, 33), (700, 3, 80), (24, 30, 5)],
])
def test_batch_tile_edges(prec, cut, shapes):
    print(f"[gpu-case] batch tiles {prec}, cut {cut}, {shapes}", flush=True)
    rng = np.random.default_rng(shapes[0][0])
    single = prec == "fp32"
    with jk.Batch(*zip(*shapes), jk.PREC_FP32 if single else jk.PREC_FP64) as b:
        b.set_config(cut, 3)
        ref = []
        for i, (n, na, no) in enumerate(shapes):
            B = rng.standard_normal((n * (n + 1) // 2, na)) / np.sqrt(na)
            c = rng.standard_normal((n, no)) / np.sqrt(n)
            occ = rng.uniform(0.2, 2.0, no)
            if no > 3:
                occ[1], occ[2] = -0.4, 0.0
            d = (c * occ) @ c.T
            b.set_rimatr(i, np.asfortranarray(B))
            b.set_inputs(i, d, c, occ)
            ref.append((orc.vj_upper_rimatr(B, [d], 1, 1.0)[0], orc.vk_upper_occ(B, True, [c], [no - 1], [occ], 1, -0.5)[0]))
        for _ in range(2):
            b.run(1.0, -0.5)
            b.synchronize()
        for i, (j, k) in enumerate(ref):
            vj, vk = b.get_outputs(i)
            assert np.abs(vk - k).max() <= (2e-5 * np.abs(k).max() if single else 1e-11), (i, shapes[i])
            assert np.abs(vj - j).max() <= (1e-6 * np.abs(j).max() if single else 1e-11), (i, shapes[i])
