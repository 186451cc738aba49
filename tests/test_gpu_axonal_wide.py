"""Axonal layers past 256 neurons -- the scatter of arriving spikes (``axwide.hip``) and the
blocked reverse scan without offsets (``hybblock.hip``) -- against the oracle, at their edges:
one neuron past a wave or a group, two and four neurons per lane, up to 640 and 1,000 neurons
(with a window in and past the blocked scan's LDS), two, four and eight taps, one, two and four
history words, a last partial block of steps, more than 64 arrivals in a step, one step, and the
neuron's options; and the dense scans, which keep learned spreads, hard taps and more taps (past
8 forward, 12 backward). Tolerances: ``tests/helpers.py``."""

import ctypes

import pytest
import torch

from helpers import gen
from test_gpu_axonal import _check_case
from test_gpu_modes import test_hard_tap_modes_match_oracle as check_hard_taps

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
    (15, 1, 1000, 4.0, 0.5, {'bias': True}),
    # the dense forward: 11 taps, a spread per source; and the dense backward: 13 taps, a spread
    (20, 2, 300, 9.0, 4.2, {}),
    (20, 2, 290, 9.0, 5.5, {'drop': True}),
    (19, 2, 300, 10.0, 0.7, {'sig_p': True}),
    (17, 1, 515, 12.0, 3.0, {'sig_p': True, 'bias': True}),
    (80, 1, 270, 66.0, 0.5, {'sig_p': True}),
]


@pytest.mark.gpu
@pytest.mark.parametrize('case', CASES, ids=[f'T{c[0]}N{c[2]}d{c[3]}s{c[4]}{"".join(c[5])}' for c in CASES])
def test_wide_axonal_matches_oracle(dev, case, monkeypatch):
    _check_case(dev, case, monkeypatch)


# the hard-tap forwards (dense) and their straight-through and soft backwards
HARD = [
    ('triton_approx', True, 'approx', 20, 2, 300, 12.0, 0.6),
    ('triton_ste', True, 'ste_round', 20, 2, 290, 9.0, 0.5),
    ('triton_ste', False, 'ste_interp', 20, 2, 300, 9.0, 1.0),
]


@pytest.mark.gpu
@pytest.mark.parametrize('case', HARD, ids=[c[2] for c in HARD])
def test_wide_axonal_hard_taps_match_oracle(dev, case):
    check_hard_taps(dev, case)


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


def _abi(dev, T, B, N, L, sigma, per_source, g, d, drive=0.3, grid=0):
    """Forward and backward through the C ABI; ``per_source``: the half-width as a vector, which
    takes the dense scans. ``drive``: the input's mean; ``grid``: W on multiples of 1 / grid."""
    from delrec import _lib
    lib = _lib.load()
    x, gy = (torch.randn(T, B, N, generator=g) * 1.2 + drive).to(dev), torch.randn(T, B, N, generator=g).to(dev)
    W, d = (torch.randn(N, N, generator=g) / N ** 0.5).to(dev), d.to(dev)
    if grid:
        W, x = (W * grid).round() / grid, (x * grid).round() / grid
    s = torch.full((N,), 1.0 + sigma, device=dev) if per_source else None
    lif = _lib.make_lif(2.0, 1.0, 0.0, False, False, 1, 1.0, 2.0)
    y, u, z, dx = (torch.empty(T, B, N, device=dev) for _ in range(4))
    bits = torch.empty(B, (T + 31) // 32, N, device=dev, dtype=torch.int32)
    dW, db, dd = torch.empty(N, N, device=dev), torch.empty(N, device=dev), torch.empty(N, device=dev)
    ws = [_lib.workspace(k, T, B, N, L, 0, dev) for k in (_lib.WS_AXONAL_FWD, _lib.WS_AXONAL_BWD)]
    both = dict(T=T, B=B, N=N, L=L, W=_lib.ptr(W), w_bf16=0, d=_lib.ptr(d), s=_lib.ptr(s), s_uniform=1.0 + sigma,
                drop=None, lif=lif, u=_lib.ptr(u), z=_lib.ptr(z), bits=_lib.ptr(bits))
    fwd = _lib.AxonalFwdArgs(x=_lib.ptr(x), bias=None, taps=0, y=_lib.ptr(y), rec=None, workspace=_lib.ptr(ws[0]),
                             workspace_bytes=ws[0].numel(), **both)
    bwd = _lib.AxonalBwdArgs(gy=_lib.ptr(gy), mode=_lib.DELREC_BWD_SOFT, lag=None, dx=_lib.ptr(dx), dW=_lib.ptr(dW),
                             db=_lib.ptr(db), dd=_lib.ptr(dd), ds=None, workspace=_lib.ptr(ws[1]),
                             workspace_bytes=ws[1].numel(), **both)
    assert lib.delrec_axonal_fwd(ctypes.byref(fwd), _lib.stream_of(x)) == 0
    assert lib.delrec_axonal_bwd(ctypes.byref(bwd), _lib.stream_of(x)) == 0
    torch.cuda.synchronize()
    return y, {'dx': dx, 'dW': dW, 'db': db, 'dd': dd}


@pytest.mark.gpu
@pytest.mark.parametrize('sigma', [0.0, 1.0, 3.0])
def test_wide_axonal_window_cuts_the_taps(dev, sigma):
    """Delays past the window L: taps at lags 1 .. L - 1 only, as in the dense scans (the same
    sums in another order: 1e-5 of the largest value)."""
    T, B, N, L = 40, 2, 300, 12
    d = torch.rand(N, generator=gen(5)) * 24.0 - 1.0
    y, got = _abi(dev, T, B, N, L, sigma, False, gen(3), d)
    yd, dense = _abi(dev, T, B, N, L, sigma, True, gen(3), d)
    assert torch.equal(y, yd)
    for k in got:
        torch.testing.assert_close(got[k], dense[k], rtol=1e-4, atol=1e-5 * float(dense[k].abs().max()), msg=k)


@pytest.mark.gpu
@pytest.mark.parametrize('sigma', [0.0, 1.0, 3.0])
@pytest.mark.parametrize('drive', [0.3, 4.0])
def test_wide_axonal_arrivals_at_dense_firing(dev, sigma, drive):
    """From a few arrivals a step to most sources at once (several rounds of 64, remainders of 16
    and 8). With dyadic weights, inputs and delays the recurrent sums are exact in any order, so
    the spikes are the dense scan's."""
    T, B, N, L = 50, 2, 330, 30
    d = (torch.floor(torch.rand(N, generator=gen(5)) * 20 * 16) + 0.5) / 16
    y, _ = _abi(dev, T, B, N, L, sigma, False, gen(3), d, drive, 4096)
    yd, _ = _abi(dev, T, B, N, L, sigma, True, gen(3), d, drive, 4096)
    assert torch.equal(y, yd)
    assert float(y.mean()) > (0.6 if drive > 1 else 0.05)


@pytest.mark.gpu
def test_wide_axonal_steps_past_4_gib(dev):
    """A (B, N) step of more than 4 GiB: past the 32-bit offsets of the scans above. With one step
    and no spike before it, u = x, y = [x >= 1] and dx = gy sg(x - 1)."""
    from delrec import _lib
    lib = _lib.load()
    B, N, L = 3_600_000, 300, 8
    print(f'B={B} N={N}: {B * N * 4 / 2 ** 30:.2f} GiB a step', flush=True)
    g = torch.Generator(dev).manual_seed(1)
    x = torch.randn(1, B, N, generator=g, device=dev)
    W, d = torch.randn(N, N, generator=g, device=dev), torch.rand(N, generator=g, device=dev) * 4
    y, u, z = (torch.full_like(x, 7.0) for _ in range(3))
    bits = torch.empty(B, 1, N, device=dev, dtype=torch.int32)
    lif = _lib.make_lif(2.0, 1.0, 0.0, False, False, 1, 1.0, 2.0)
    both = dict(T=1, B=B, N=N, L=L, W=_lib.ptr(W), w_bf16=0, d=_lib.ptr(d), s=None, s_uniform=1.5, drop=None, lif=lif,
                u=_lib.ptr(u), bits=_lib.ptr(bits))
    ws = _lib.workspace(_lib.WS_AXONAL_FWD, 1, B, N, L, 0, dev)
    fwd = _lib.AxonalFwdArgs(x=_lib.ptr(x), bias=None, taps=0, y=_lib.ptr(y), rec=None, z=_lib.ptr(z),
                             workspace=_lib.ptr(ws), workspace_bytes=ws.numel(), **both)
    assert lib.delrec_axonal_fwd(ctypes.byref(fwd), _lib.stream_of(x)) == 0
    assert torch.equal(u, x) and torch.equal(y, (x >= 1).float()) and float(z.abs().max()) == 0
    del ws, z
    gy = y.add_(0.5)
    dx = torch.full_like(x, 7.0)
    ws = _lib.workspace(_lib.WS_AXONAL_BWD, 1, B, N, L, 0, dev)
    bwd = _lib.AxonalBwdArgs(gy=_lib.ptr(gy), z=None, mode=_lib.DELREC_BWD_SOFT, lag=None, dx=_lib.ptr(dx), dW=None,
                             db=None, dd=None, ds=None, workspace=_lib.ptr(ws), workspace_bytes=ws.numel(), **both)
    assert lib.delrec_axonal_bwd(ctypes.byref(bwd), _lib.stream_of(x)) == 0
    # the surrogate's alpha / 2 / (1 + (pi / 2 alpha (u - 1))^2) at alpha = 2
    ref = gy.div_(x.sub_(1.0).mul_(torch.pi).square_().add_(1.0))
    assert float(dx.sub_(ref).abs_().max()) < 1e-5
