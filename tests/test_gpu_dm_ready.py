"""rjk_vk_upper_dm_dev returns with its result in place: read at once on another stream, with no wait in
between (the context's own stream does not synchronise with the reader's), on each of its routes: a
low-rank density, an indefinite one, one that is not symmetric, a zero one.  Exact: the same numbers after a wait;
against the host entry point 1e-11, as tests/test_gpu_jk.py."""
import numpy as np
import pytest
import torch

from rest_amd import jk

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind", ["low rank", "indefinite", "general", "zero"])
@pytest.mark.parametrize("ns", [1, 2])
def test_result_ready_on_return(kind, ns):
    print(f"[gpu-case] density-only K ready on return: {kind}, {ns} spins", flush=True)
    n, naux = 300, 1200
    rng = np.random.default_rng(ns)
    ds = []
    for _ in range(ns):
        q = np.linalg.qr(rng.standard_normal((n, n)))[0]
        d = {"low rank": 2 * q[:, :40] @ q[:, :40].T, "indefinite": (q * np.linspace(-1, 1, n)) @ q.T,
             "general": rng.standard_normal((n, n)), "zero": np.zeros((n, n))}[kind]
        ds.append(d if kind == "general" else 0.5 * (d + d.T))
    dm = torch.from_numpy(np.stack([np.ascontiguousarray(d.T) for d in ds])).cuda()
    out = torch.empty((ns, n * (n + 1) // 2), dtype=torch.float64, device="cuda")
    with jk.DeviceRI(n, naux) as r:
        r.fill_synthetic(7)
        ref = r.vk_dm(ds, ns, -0.5)
        other = torch.cuda.Stream()
        with torch.cuda.stream(other):
            out.fill_(float("nan"))
            other.synchronize()
            r.vk_dm_dev(dm.data_ptr(), ns, -0.5, out.data_ptr())
            first = out.clone()          # on `other`: nothing orders it after the context's stream but the return
            other.synchronize()
        r.synchronize()
        torch.cuda.synchronize()
        assert torch.equal(first, out)
        assert np.abs(out.cpu().numpy() - ref).max() <= 1e-11
