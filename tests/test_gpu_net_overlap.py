"""The network's forward pass with its output over its input: the same array, and shifted by some rows either way,
with no hidden layer (one product, which reads rows while it writes others) and with one.  Exact: the
same bits as into an array of its own."""
import pytest
import torch

from rest_amd import learned as lg

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("layers", [0, 1])
@pytest.mark.parametrize("n_in,n_out", [(96, 96), (130, 70), (64, 200)])
@pytest.mark.parametrize("shift", [0, 64, -64])
def test_output_over_input(layers, n_in, n_out, shift):
    batch = 1000
    print(f"[gpu-case] forward {n_in}->{n_out}, {layers} hidden layers, output {shift} floats off", flush=True)
    net = lg.Net(n_in, n_out, 48, layers, batch, seed=5)
    x = torch.randn((batch, n_in), generator=torch.Generator().manual_seed(1)).cuda()
    ref = torch.empty((batch, n_out), device="cuda")
    torch.cuda.synchronize()
    net.forward_dev(x, ref)
    buf = torch.zeros(64 + batch * max(n_in, n_out) + 64, device="cuda")
    xs = buf[64:64 + batch * n_in].view(batch, n_in)
    xs.copy_(x)
    ys = buf[64 + shift:64 + shift + batch * n_out].view(batch, n_out)
    torch.cuda.synchronize()
    net.forward_dev(xs, ys)
    assert torch.equal(ys, ref)
    net.close()
