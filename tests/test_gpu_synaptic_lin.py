"""The synaptic reverse scan on interpolation tables (``synlin.hip``) against the float64 oracle, at
its edges: one source block and a partial one, one receiver slice and several, windows at the
limits of the 32 and 64 slot tables, half-widths that are whole numbers and that are not, delays
on the integers, just below one (a fraction that rounds up) and below 0, where whole runs of
lags fall away. Tolerances: ``tests/helpers.py``."""

import pytest
import torch

from helpers import check_grads, first_flip, gen, grad_eps, lif_params, oracle_synaptic, syn_budget
from test_gpu_synaptic import SYN_CASES, test_synaptic_fwd_bwd_matches_oracle as check_case

CASES = [
    # T, B, N, delays from, to, sigma, options
    (20, 2, 16, 0.0, 9.0, 0.0, ()),
    (33, 2, 63, 0.0, 26.0, 1.0, ('bias', 'drop')),
    (34, 2, 65, 0.0, 26.9, 0.0, ('integer',)),
    (24, 2, 70, -7.0, 8.0, 1.0, ()),
    (24, 2, 40, -3.0, 12.0, 0.5, ()),
    (40, 1, 130, 0.0, 30.0, 0.4, ()),
    (44, 1, 100, 0.0, 55.0, 1.0, ('bf16',)),
    (70, 1, 48, 0.0, 40.0, 2.7, ()),
    (30, 1, 256, 0.0, 16.0, 3.0, ()),
    (22, 1, 257, 0.0, 20.0, 1.0, ('detach',)),
    (18, 1, 520, 0.0, 12.0, 0.0, ()),
]


@pytest.mark.gpu
@pytest.mark.parametrize('case', CASES, ids=[f'T{c[0]}N{c[2]}d{c[3]}_{c[4]}s{c[5]}{"".join(c[6])}' for c in CASES])
def test_interpolated_backward_matches_oracle(dev, case):
    from delrec.kernels import EventDrivenSyn
    from delrec.neuron import ATan, LIFNode
    T, B, N, lo, hi, sigma, opts = case
    print(f'case {case}', flush=True)
    g = gen(11)
    x = torch.randn(T, B, N, generator=g) * 1.2 + 0.3
    W = torch.randn(N, N, generator=g) * (1.5 / N ** 0.5)
    bf16 = 'bf16' in opts
    if bf16:
        W = W.bfloat16().float()
    d = lo + torch.rand(N, N, generator=g) * (hi - lo)
    if 'integer' in opts:
        d = d.floor()
        d.view(-1)[::5] = d.view(-1)[::5] + (1.0 - 2.0 ** -24)      # (rounds to the next integer past 1)
        d.view(-1)[::7] = 1.0 - 2.0 ** -24
    gy = torch.randn(T, B, N, generator=g)
    bias = torch.randn(N, generator=g) * 0.1 if 'bias' in opts else None
    drop = (torch.rand(B, N, generator=g) > 0.2).float() / 0.8 if 'drop' in opts else None
    detach = 'detach' in opts
    lif = lif_params(detach_reset=detach)

    class Cfg:
        surrogate_function, surrogate_gamma, detach_reset, recurrent_dropout_rate = ATan(2.0), 1.0, detach, 0.0

    class Layer:
        config = Cfg()
        neuron_module = LIFNode(tau=2.0, decay_input=False, v_threshold=1.0, v_reset=0.0, detach_reset=detach)
        use_sig_p, p_spread, round_delays, training = False, None, False, False

    layer = Layer()
    layer.sigma = sigma
    y_ref, u_ref, gref = oracle_synaptic(x, W, d, lif, sigma, gy, bias=bias, drop=drop)
    xg = x.to(dev).requires_grad_(True)
    Wg = (W.bfloat16() if bf16 else W).to(dev).requires_grad_(True)
    dg = d.to(dev).requires_grad_(True)
    bg = None if bias is None else bias.to(dev).requires_grad_(True)
    y = EventDrivenSyn.apply(xg, Wg, dg, torch.zeros(N, device=dev), bg, None if drop is None else drop.to(dev), layer)
    (y * gy.to(dev)).sum().backward()
    torch.cuda.synchronize()
    flip = first_flip(y.detach().cpu(), y_ref, u_ref, lif.v_threshold)
    assert flip is None, f'near-threshold flip at t={flip}'
    _, _, g64 = oracle_synaptic(x, W, d, lif, sigma, gy, bias=bias, drop=drop, dtype=torch.float64, forced=y.detach().cpu())
    got = {'x': xg.grad, 'W': Wg.grad.float(), 'd': dg.grad}
    if bg is not None:
        got['bias'] = bg.grad
    plain = drop is None
    check_grads(got, g64, gref, 2e-2 if bf16 else 1e-4, 1e-5, eps=grad_eps(bf16),
                budget=syn_budget(g64['x'], y.detach().cpu(), d, sigma, W=W) if plain else None)


# the gather per tap, which keeps the spreads per source and the layers whose tables miss LDS, at each
# of its compiled tap runs (4, 8, 12) and a runtime count; the last two take it without the switch
GATHER = [SYN_CASES[i] for i in (0, 1, 2, 7, 8)] + [
    (14, 2, 40, 6.0, 0.3, {'sig_p': True}),
    (14, 2, 72, 6.0, 4.0, {'sig_p': True, 'bias': True}),
]


@pytest.mark.gpu
@pytest.mark.parametrize('case', GATHER, ids=[f'N{c[2]}s{c[4]}{"".join(c[5])}' for c in GATHER])
def test_gather_per_tap_backward_matches_oracle(dev, case, monkeypatch):
    monkeypatch.setenv('DELREC_SYN_LIN', '0')
    check_case(dev, case)


@pytest.mark.gpu
def test_interpolated_backward_on_delays_and_weights_that_are_no_numbers(dev, monkeypatch):
    """A NaN delay has no lag of positive weight, and a connection without one is its weight times
    0 (an infinite weight: NaN in its source's column), as in the gather per tap."""
    from delrec import _lib
    from delrec.kernels.synaptic_eventdriven import syn_backward, syn_forward
    T, B, N, sigma = 19, 2, 48, 1.0
    g = gen(3)
    x, gy = (torch.randn(T, B, N, generator=g).to(dev) for _ in range(2))
    W, d = (torch.randn(N, N, generator=g) / N ** 0.5).to(dev), (torch.rand(N, N, generator=g) * 9).to(dev)
    lif = _lib.make_lif(2.0, 1.0, 0.0, False, False, 1, 1.0, 2.0)
    y, u, bits, L, _, _, s_max, _ = syn_forward(x, W, d, None, None, None, 1 + sigma, d, None, None, lif)
    W, d = W.clone(), d.clone()
    d[3, 5] = float('nan')

    def both():
        out = []
        for switch in ('1', '0'):
            monkeypatch.setenv('DELREC_SYN_LIN', switch)
            out.append(syn_backward(gy, u, y, bits, W, 0, d, None, None, None, 1 + sigma, s_max, None, lif, L,
                                    False, False, False, False)[0])
        return out

    got, ref = both()
    assert not torch.equal(got, ref), 'the tables and the gather sum in another order'
    assert bool(ref.isfinite().all())
    torch.testing.assert_close(got, ref, rtol=1e-4, atol=1e-5)
    W[7, 9], d[7, 9] = float('inf'), -30.0
    for dx in both():
        assert bool(dx[:, :, 9].isnan().all())
        assert bool(dx[-1, :, :9].isfinite().all()) and bool(dx[-1, :, 10:].isfinite().all())
