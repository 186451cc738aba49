"""The plain LIF layer's blocks of loaded steps (16 forward, 8 backward), at step counts around
their multiples, against the oracle; and its form of one load at a time (short runs forward,
layers of many waves) against the blocks, bit for bit. Elementwise: the forward's operations are the oracle's own,
the gradients differ by the rounding of the surrogate's division (1e-6 relative)."""

import pytest
import torch

from helpers import gen, lif_params
from oracle import scans


@pytest.mark.gpu
@pytest.mark.parametrize('T', [1, 7, 8, 9, 15, 16, 17, 23, 24, 25, 31, 32, 33, 49])
def test_lif_layer_step_counts(dev, T):
    from delrec.neuron import LIFNode
    g = gen(T)
    x, gy = torch.randn(T, 3, 37, generator=g) * 0.8, torch.randn(T, 3, 37, generator=g)
    xr = x.clone().requires_grad_(True)
    y_ref, _ = scans.lif_layer(xr, lif_params())
    y_ref.backward(gy)
    xg = x.to(dev).requires_grad_(True)
    y = LIFNode(tau=2.0, decay_input=False, step_mode='m')(xg)
    y.backward(gy.to(dev))
    assert torch.equal(y.detach().cpu(), y_ref.detach())
    torch.testing.assert_close(xg.grad.cpu(), xr.grad, rtol=1e-5, atol=1e-6)


@pytest.mark.gpu
@pytest.mark.parametrize('T,B,N', [(25, 257, 511), (3, 1024, 513), (100, 256, 1025), (99, 256, 1024)])
def test_lif_layer_of_many_waves_equals_its_slices(dev, T, B, N):
    from delrec.neuron import LIFNode
    lif = LIFNode(tau=2.0, decay_input=False, step_mode='m')
    g = torch.Generator(dev).manual_seed(T)
    x, gy = (torch.randn(T, B, N, generator=g, device=dev) for _ in range(2))

    def run(x, gy):
        x = x.clone().requires_grad_(True)
        y = lif(x)
        y.backward(gy)
        return y.detach(), x.grad

    whole = run(x, gy)
    for b in (0, B // 2, B - 2):
        for a, c in zip(run(x[:, b:b + 2].contiguous(), gy[:, b:b + 2].contiguous()), whole):
            assert torch.equal(a, c[:, b:b + 2])
