"""A backward workspace that ends before the blocked or the interpolated scan's operands (as a
caller holds that was told its size without them): the call runs in the form that needs none,
bit for bit what the switch that names that form gives; one short of that form too is refused."""

import pytest
import torch

from helpers import gen
from test_gpu_synaptic import _Layer, hybrid_layer, lif_params

CASES = {'hybrid': ('DELREC_SYN_BWD_HYB', 100, 1.0), 'synaptic': ('DELREC_SYN_LIN', 100, 1.0)}


def _run(kind, dev, sigma, N):
    from delrec.kernels import EventDrivenSyn
    g = gen(9)
    T, B = 23, 3
    W = torch.randn(N, N, generator=g) / N ** 0.5
    x, gy = torch.randn(T, B, N, generator=g).to(dev), torch.randn(T, B, N, generator=g).to(dev)
    x.requires_grad_(True)
    if kind == 'hybrid':
        layer = hybrid_layer(N, W, torch.rand(N, generator=g) * 15, torch.randint(5, (N, N), generator=g).float(), dev,
                             sigma_init=sigma)
        layer(x).backward(gy)
        return [x.grad] + [p.grad for p in layer.parameters()]
    leaves = [W.to(dev).requires_grad_(True), (torch.rand(N, N, generator=g) * 15).to(dev).requires_grad_(True)]
    EventDrivenSyn.apply(x, *leaves, torch.zeros(N, device=dev), None, None, _Layer(sigma, lif_params())).backward(gy)
    return [x.grad] + [t.grad for t in leaves]


@pytest.mark.gpu
@pytest.mark.parametrize('kind', CASES)
def test_workspace_without_the_packed_operands_takes_another_form(dev, kind, monkeypatch):
    from delrec import _lib
    switch, N, sigma = CASES[kind]
    own = _run(kind, dev, sigma, N)
    with monkeypatch.context() as m:
        m.setenv(switch, '0')
        general = _run(kind, dev, sigma, N)
    assert not torch.equal(own[0], general[0]), 'the case must take the packed form by default'
    # the packed operands: hybrid 20 bytes a connection, padded to 64 receivers and 16 sources,
    # and two ints a source; synaptic 8 bytes a connection, padded to 16 receivers and 64 sources
    pad = lambda n, m: -(-n // m) * m
    extra = (pad(16 * pad(N, 64) // 4 * pad(N, 16), 256) + pad(pad(N, 64) * pad(N, 16), 256) + pad(8 * N, 256)
             if kind == 'hybrid' else pad(8 * pad(N, 16) * pad(N, 64), 256))
    real = _lib.workspace

    def shorter(by):
        return lambda k, *a: real(k, *a)[:-by] if k == _lib.WS_SYN_BWD else real(k, *a)

    for by in (1, extra):
        monkeypatch.setattr(_lib, 'workspace', shorter(by))
        for a, b in zip(_run(kind, dev, sigma, N), general):
            assert torch.equal(a, b)
    monkeypatch.setattr(_lib, 'workspace', shorter(extra + 1))
    with pytest.raises(_lib.DelrecError):
        _run(kind, dev, sigma, N)
