"""Axonal layers past 256 neurons -- the scatter of arriving spikes (``axwide.hip``) and the
blocked reverse scan without offsets (``hybblock.hip``) -- against the oracle, at their edges:
one neuron past a wave or a group, two and four neurons per lane, up to 640 and 1,000 neurons
(the latter's window past the blocked scan's LDS), two, four and eight taps, one, two and four
history words, a last partial block of steps, more than 64 arrivals in a step, one step, and the
neuron's options. Tolerances: ``tests/helpers.py``."""

import pytest
import torch

from helpers import gen
from test_gpu_axonal import _check_case

CASES = [
    # T, B, N, dmax, sigma, extra
    (21, 2, 257, 6.0, 0.0, {}),
    (22, 2, 273, 14.0, 1.0, {'bias': True}),
    (23, 1, 384, 24.0, 3.0, {}),
    (26, 2, 385, 30.0, 0.4, {'drop': True, 'bias': True}),
    (19, 1, 512, 9.0, 1.0, {'soft': True}),
    (20, 2, 513, 12.0, 0.0, {'detach': True}),
    (18, 1, 640, 20.0, 1.3, {'decay_input': True}),
    (14, 1, 1000, 26.0, 0.5, {}),
    (90, 1, 260, 75.0, 1.0, {'triangle': True}),
    (150, 1, 258, 140.0, 0.0, {'v_reset': -0.2}),
    (1, 2, 300, 5.0, 1.0, {}),
]


@pytest.mark.gpu
@pytest.mark.parametrize('case', CASES, ids=[f'T{c[0]}N{c[2]}d{c[3]}s{c[4]}{"".join(c[5])}' for c in CASES])
def test_wide_axonal_matches_oracle(dev, case, monkeypatch):
    _check_case(dev, case, monkeypatch)


@pytest.mark.gpu
def test_wide_axonal_repeats_bit_for_bit(dev):
    """Two passes on the same inputs: arrivals and partial sums are taken in a fixed order."""
    from delrec.kernels import AxonalRecdelHip
    g = gen(1)
    T, B, N = 40, 6, 320
    x, gy = (torch.randn(T, B, N, generator=g).to(dev) for _ in range(2))
    W, d = (torch.randn(N, N, generator=g) / N ** 0.5).to(dev), (torch.rand(N, generator=g) * 18).to(dev)
    out = []
    for _ in range(2):
        xs, Ws, ds = (t.clone().requires_grad_(True) for t in (x, W, d))
        y = AxonalRecdelHip.apply(xs, Ws, None, ds, torch.zeros(N, device=dev), None, 1.0, 2.0, 1.0, 0.0, False, False,
                                  1, 1.0, False, 0, 2.0)
        y.backward(gy)
        out.append([y.detach(), xs.grad, Ws.grad, ds.grad])
    for a, b in zip(*out):
        assert torch.equal(a, b)
