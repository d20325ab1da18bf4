"""GPU parity of the batched BF16 half-transform at the edges of its units: nbf around a 16-row fragment and
a 32-deep step, column counts around 32, 96 and 192 (one tile, two, three), auxiliary counts that leave
waves of a work-group without a unit.  K with three planes against the float64 oracle: 2e-6 of the largest
element (FP32 level, as tests/test_gpu_kbf.py); J against it: 1e-6 (B held in FP32, FP64 sums)."""
import numpy as np
import pytest

from oracle import oracle as orc
from rest_amd import jk

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shapes", [
    [(1, 1, 1), (15, 9, 4), (16, 8, 16), (17, 7, 3)],
    [(31, 13, 31), (32, 33, 32), (33, 5, 33), (48, 16, 40)],
    [(96, 11, 96), (97, 3, 97), (65, 21, 64), (130, 10, 65)],
    [(200, 5, 193), (257, 3, 129)],
])
def test_batch_half_transform_edges(shapes):
    print(f"[gpu-case] batch edges {shapes}", flush=True)
    rng = np.random.default_rng(len(shapes) * 97 + shapes[0][0])
    with jk.Batch(*zip(*shapes), jk.PREC_BF16X3) as b:
        ref = []
        for i, (n, na, no) in enumerate(shapes):
            B = rng.standard_normal((n * (n + 1) // 2, na)) / np.sqrt(na)
            c = rng.standard_normal((n, no)) / np.sqrt(n)
            occ = rng.uniform(0.2, 2.0, no)
            if no > 2:
                occ[1] = -0.4
            d = (c * occ) @ c.T
            b.set_rimatr(i, np.asfortranarray(B))
            b.set_inputs(i, d, c, occ)
            ref.append((orc.vj_upper_rimatr(B, [d], 1, 1.0)[0], orc.vk_upper_occ(B, True, [c], [no - 1], [occ], 1, -0.5)[0]))
        for _ in range(2):
            b.run(1.0, -0.5)
            b.synchronize()
        for i, (j, k) in enumerate(ref):
            vj, vk = b.get_outputs(i)
            assert np.abs(vk - k).max() <= 2e-6 * np.abs(k).max(), (i, shapes[i])
            assert np.abs(vj - j).max() <= 1e-6 * np.abs(j).max(), (i, shapes[i])
