"""The network's loss and gradient at the edges of its GEMM tiles (64 rows, 64 columns, 64-deep blocks,
batch splits of 256 rows) against the MLP oracle.  Bounds as tests/test_gpu_learned.py: loss 1e-5,
each layer's gradient 5e-3 in relative norm (BF16 operands; flips of intermediate roundings)."""
import numpy as np
import pytest
import torch

from oracle import mlp_oracle as mo
from rest_amd import learned as lg

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dims,batch", [
    ((5, 17, 2, 1), 1), ((64, 64, 1, 64), 65), ((65, 33, 3, 3), 257), ((130, 96, 2, 70), 513), ((33, 128, 0, 1), 300),
    ((219, 256, 3, 196), 4097),
])
def test_gradient_at_tile_edges(dims, batch):
    n_in, hidden, layers, n_out = dims
    print(f"[gpu-case] network {dims} batch {batch}", flush=True)
    rng = np.random.default_rng(batch)
    net = lg.Net(n_in, n_out, hidden, layers, max(batch, 64), seed=3)
    net.set_params((net.get_params() + 0.05 * rng.standard_normal(net.nparam)).astype(np.float32))
    X = rng.standard_normal((batch, n_in)).astype(np.float32)
    T = rng.standard_normal((batch, n_out)).astype(np.float32)
    M = (rng.random((batch, n_out)) > 0.4).astype(np.float32)
    M[0, 0] = 1.0
    dev = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()
    loss, g = net.loss_grad_dev(dev(X), dev(T), dev(M), want_grad=True)
    lo, go = mo.loss_grad(net.get_params(), net.dims, X, T, M, bf16=True)
    assert abs(loss - lo) <= 1e-5 * abs(lo)
    off = 0
    for din, dout in zip(net.dims[:-1], net.dims[1:]):
        for cnt in (din * dout, dout):
            a, b = g[off:off + cnt], go[off:off + cnt]
            assert np.linalg.norm(a - b) <= 5e-3 * np.linalg.norm(b) + 1e-12
            off += cnt
