"""The blocked reverse scan of hybrid delays (``hybblock.hip``) against the float64 oracle, at
the sizes where its groups, chunks, blocks and ring runs have edges: one group and a partial
one, a quarter of the receivers more and less than whole chunks of 16, one, two and four
neurons per lane, far groups dealt out over more than one round; early runs of 2, 4 and 8
slots (half-widths over 1 near the delay 0, negative bases), more than 9 offsets (the wider
ring), every source near, steps that are no multiple of a block, tap counts past four; and,
with a dropout mask and a bias, against the per-tap gather. Tolerances: ``tests/helpers.py``."""

import pytest
import torch

from test_gpu_synaptic import test_hybrid_fwd_bwd_matches_oracle as check_case
from test_gpu_synaptic import hybrid_layer
from helpers import gen

CASES = [
    # T, B, N, base range, max offset, bf16 weights, sigma
    (21, 2, 16, (0.0, 9.0), 4, False, 1.0),
    (22, 3, 17, (0.0, 14.0), 3, True, 1.0),
    (23, 2, 63, (0.0, 24.0), 8, True, 3.0),
    (24, 2, 65, (-3.0, 12.0), 2, False, 3.0),       # early runs of 8
    (25, 2, 130, (0.0, 30.0), 11, False, 1.0),      # 12 offsets: the ring of 32 slots
    (26, 2, 192, (0.0, 2.5), 4, False, 0.0),        # every source near
    (27, 2, 193, (0.0, 26.0), 4, True, 0.4),
    (28, 2, 256, (0.0, 33.0), 8, False, 1.0),
    (29, 2, 257, (0.0, 20.0), 4, False, 0.0),
    (30, 2, 385, (0.0, 28.0), 5, True, 2.5),
    (31, 1, 513, (0.0, 18.0), 3, False, 1.0),
    (22, 1, 600, (0.0, 12.0), 2, True, 0.0),
    (18, 1, 800, (0.0, 6.0), 3, True, 1.0),
    (18, 1, 1024, (0.0, 4.0), 2, False, 1.0),       # the limit
    (20, 2, 48, (0.0, 10.0), 3, False, 4.0),        # ten taps
]


@pytest.mark.gpu
@pytest.mark.parametrize('case', CASES, ids=[f'T{c[0]}N{c[2]}K{c[4]}{"bf16" if c[5] else ""}s{c[6]}' for c in CASES])
def test_blocked_backward_matches_oracle(dev, case):
    check_case(dev, case)


@pytest.mark.gpu
@pytest.mark.parametrize('N', [96, 260])
def test_blocked_backward_repeats_bit_for_bit(dev, N):
    """Two passes on the same inputs: partial sums meet in a fixed order."""
    g = gen(3)
    T, B = 33, 5
    layer = hybrid_layer(N, torch.randn(N, N, generator=g) / N ** 0.5, torch.rand(N, generator=g) * 20,
                         torch.randint(5, (N, N), generator=g).float(), dev, bf16=False, sigma_init=1.0)
    x, gy = torch.randn(T, B, N, generator=g).to(dev), torch.randn(T, B, N, generator=g).to(dev)
    out = []
    for _ in range(2):
        layer.zero_grad(set_to_none=True)
        xi = x.clone().requires_grad_(True)
        layer(xi).backward(gy)
        out.append([xi.grad] + [p.grad for p in layer.parameters()])
    for a, b in zip(*out):
        assert torch.equal(a, b)


@pytest.mark.gpu
def test_blocked_backward_with_dropout_and_bias(dev, monkeypatch):
    """The same pass through ``syn_bwd_kernel``: the sums differ by their order (up to N terms of
    2^-24 each; 1e-5 of the largest value)."""
    from delrec.kernels import HybridSynDelay
    g = gen(4)
    T, B, N = 27, 3, 200
    layer = hybrid_layer(N, torch.randn(N, N, generator=g) / N ** 0.5, torch.rand(N, generator=g) * 15,
                         torch.randint(6, (N, N), generator=g).float(), dev, bf16=False, sigma_init=1.0)
    drop = (torch.rand(B, N, generator=g) > 0.3).float().to(dev) / 0.7
    x, gy = torch.randn(T, B, N, generator=g).to(dev), torch.randn(T, B, N, generator=g).to(dev)
    bias = (torch.randn(N, generator=g) * 0.1).to(dev)
    out = []
    for off in (False, True):
        if off:
            monkeypatch.setenv('DELREC_SYN_BWD_HYB', '0')
        layer.zero_grad(set_to_none=True)
        xi, bi = x.clone().requires_grad_(True), bias.clone().requires_grad_(True)
        HybridSynDelay.apply(xi, layer.recurrent_weights, layer.recurrent_delays, bi, drop, layer).backward(gy)
        out.append([xi.grad, bi.grad] + [p.grad for p in layer.parameters()])
    for a, b in zip(*out):
        torch.testing.assert_close(a, b, rtol=1e-4, atol=1e-5 * float(b.abs().max()))


# which backward a call takes: sources starting below lag 4 (`near`, a share) are summed step by
# step in the blocked scan, and more than 9 offsets need its ring of 32 slots, so it gives way to
# the offset-stacked scan (every lag >= 1) or the gather per tap (sigma 0.5: lags below 1)
ROUTES = [
    # N, offsets, bf16 weights, sigma, near share, expected
    (200, 12, False, 0.0, 0.1, 'offset-stacked'),
    (200, 5, False, 0.0, 0.5, 'blocked'),
    (256, 5, True, 0.0, 0.6, 'offset-stacked'),
    (256, 5, True, 0.0, 0.1, 'blocked'),
    (256, 9, True, 0.0, 0.03, 'offset-stacked'),    # 15 far groups: one past the summing waves
    (200, 12, False, 0.5, 0.6, 'gather per tap'),
    (200, 12, False, 0.5, 0.1, 'blocked'),
    (200, 5, True, 0.5, 1.0, 'blocked'),
]


@pytest.mark.gpu
@pytest.mark.parametrize('case', ROUTES, ids=[f'N{c[0]}K{c[1]}{"bf16" if c[2] else ""}s{c[3]}near{c[4]}' for c in ROUTES])
def test_backward_form_follows_the_near_share_and_the_offsets(dev, case, monkeypatch, capfd):
    N, K, bf16, sigma, near, expected = case
    monkeypatch.setenv('DELREC_LOG_PLAN', '1')
    g = gen(6)
    base = 5.0 + torch.rand(N, generator=g) * 25
    base[:round(near * N)] = torch.rand(round(near * N), generator=g) * 2
    layer = hybrid_layer(N, torch.randn(N, N, generator=g) / N ** 0.5, base,
                         torch.randint(K, (N, N), generator=g).float(), dev, bf16=bf16, sigma_init=sigma)
    x = torch.randn(12, 2, N, generator=g).to(dev).requires_grad_(True)
    layer(x).sum().backward()
    torch.cuda.synchronize()
    assert f'hybrid backward: {expected}' in capfd.readouterr().err


# a smallest delay that is too large but still below s - 1, or an offset count that is too small
# there (and, above 16 offsets, wherever the lags lie): no form may rely on them, so the
# gradients are the oracle's. (d_min, off_min, off_count) -> what the call states instead
MISSTATED = [
    ((22, 2, 200, (-4.0, 12.0), 4, False, 1.0), lambda d, o, n: (0.0, o, n)),
    ((22, 2, 48, (-6.0, 12.0), 4, True, 3.0), lambda d, o, n: (1.9, o, n)),
    ((22, 2, 200, (0.0, 30.0), 11, False, 1.0), lambda d, o, n: (d, o, 5)),
    ((22, 1, 530, (-2.0, 8.0), 3, False, 1.0), lambda d, o, n: (0.5, o, n)),
    ((30, 2, 200, (-0.5, 40.0), 16, False, 0.0), lambda d, o, n: (0.0, o, n)),
]


def _state(monkeypatch, change):
    from delrec.kernels import synaptic_eventdriven as se
    real = se.hybrid_form

    def form(d_min, s, rng):
        d, o, n = change(d_min, *rng)
        return real(d, s, (o, n))

    monkeypatch.setattr(se, 'hybrid_form', form)


@pytest.mark.gpu
@pytest.mark.parametrize('case,change', MISSTATED, ids=[f'N{c[0][2]}K{c[0][4]}s{c[0][6]}' for c in MISSTATED])
def test_blocked_backward_does_not_rely_on_a_misstated_range(dev, case, change, monkeypatch, capfd):
    _state(monkeypatch, change)
    monkeypatch.setenv('DELREC_LOG_PLAN', '1')
    check_case(dev, case)
    assert 'hybrid backward: blocked' in capfd.readouterr().err


# where every lag is said to be >= 1 (and up to 16 offsets), the scans do rely on the stated
# range: a call that breaks it gets NaN everywhere, never a wrong gradient
REFUSED = [
    ((22, 2, 200, (-0.5, 30.0), 4, False, 0.0), lambda d, o, n: (0.0, o, n)),
    ((22, 2, 256, (0.0, 30.0), 11, False, 0.0), lambda d, o, n: (d, o, 5)),
]


@pytest.mark.gpu
@pytest.mark.parametrize('case,change', REFUSED, ids=['d_min', 'offsets'])
def test_blocked_backward_refuses_a_broken_range(dev, case, change, monkeypatch, capfd):
    T, B, N, (lo, hi), K, bf16, sigma = case
    _state(monkeypatch, change)
    monkeypatch.setenv('DELREC_LOG_PLAN', '1')
    g = gen(2)
    layer = hybrid_layer(N, torch.randn(N, N, generator=g) / N ** 0.5, lo + torch.rand(N, generator=g) * (hi - lo),
                         torch.randint(K + 1, (N, N), generator=g).float(), dev, bf16=bf16, sigma_init=sigma)
    x = torch.randn(T, B, N, generator=g).to(dev).requires_grad_(True)
    layer(x).sum().backward()
    torch.cuda.synchronize()
    assert 'hybrid backward: blocked' in capfd.readouterr().err
    assert bool(x.grad.isnan().all())
