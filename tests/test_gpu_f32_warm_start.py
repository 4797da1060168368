"""float32 warm start (zero-hidden pass and all Picard passes in one launch) at
the edges of its tiles (32 steps per wave, 128 per tile) against the frozen-gate
recurrence walked in float64.

Bar: m is a sum of at most T float32 terms and n, c, h follow it through e^{z - m},
so a slot is off by at most about T u max(1, |m|) relative to its largest value
(u = 2^-24), once per pass."""

import pytest
import torch

from pararnn_amd import ops

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
EPS = 1e-6


def _walk(wx, r, h0, P):
    """Frozen-gate passes, one sequence at a time per batch row, in float64."""
    B, T, d4 = wx.shape
    d = d4 // 4
    start = torch.zeros(B, 4, d, dtype=torch.float64) if h0 is None else h0
    pre, out = wx, None
    for p in range(P + 1):
        c, n, m = start[:, 0], start[:, 1], start[:, 2]
        rows = []
        for t in range(T):
            zi, zf, zz, zo = pre[:, t].split(d, -1)
            mn = torch.maximum(zf + m, zi)
            f, i = torch.exp(zf + m - mn), torch.exp(zi - mn)
            c, n, m = f * c + i * torch.tanh(zz), f * n + i, mn
            rows.append(torch.stack((c, n, m, torch.sigmoid(zo) * c / (n + EPS)), 1))
        out = torch.stack(rows, 1)
        h = torch.cat((start[:, None, 3], out[:, :-1, 3]), 1)
        pre = wx + (r * h.unsqueeze(2)).reshape(B, T, d4)
    return out


def _check(got, want, T, P):
    for k in range(4):
        scale = want[..., k, :].abs().max().item()
        m_top = max(1.0, want[..., 2, :].abs().max().item())
        err = (got[..., k, :].double().cpu() - want[..., k, :]).abs().max().item()
        bar = (P + 1) * max(T, 8) * 2.0 ** -24 * m_top * max(scale, 1e-3) + 1e-6
        print(f"  slot {k}: err {err:.2e} bar {bar:.2e}", flush=True)
        assert err <= bar


@pytest.mark.parametrize("B,T,d", [(1, 1, 1), (2, 31, 63), (1, 32, 64), (2, 33, 65), (1, 127, 3),
                                   (1, 128, 64), (2, 129, 100), (1, 300, 64)])
@pytest.mark.parametrize("P", [0, 1, 5])
@pytest.mark.parametrize("with_h0", [False, True])
def test_rectangular(B, T, d, P, with_h0):
    g = torch.Generator().manual_seed(B * 1000 + T + d)
    wx = torch.randn(B, T, 4 * d, generator=g)
    r = torch.randn(4, d, generator=g) * 0.3
    h0 = torch.rand(B, 4, d, generator=g) if with_h0 else None
    print(f"case B={B} T={T} d={d} P={P} h0={with_h0}", flush=True)
    got = ops.slstm_init_fused(wx.to(DEV), r.to(DEV), None if h0 is None else h0.to(DEV),
                               picard_iters=P, eps=EPS)
    want = _walk(wx.double(), r.double(), None if h0 is None else h0.double(), P)
    _check(got, want, T, P)


@pytest.mark.parametrize("lengths", [[1], [27, 1, 1], [28, 29], [111, 1, 130], [5] * 40,
                                     [31, 1, 1], [32, 33], [127, 1, 130]])
@pytest.mark.parametrize("P", [0, 3])
def test_packed(lengths, P):
    d, N = 70, sum(lengths)
    g = torch.Generator().manual_seed(N + P)
    wx = torch.randn(1, N, 4 * d, generator=g)
    r = torch.randn(4, d, generator=g) * 0.3
    h0 = torch.rand(len(lengths), 4, d, generator=g)
    cu = torch.tensor([0, *torch.tensor(lengths).cumsum(0).tolist()])
    print(f"case packed {lengths} P={P}", flush=True)
    got = ops.slstm_init_fused(wx.to(DEV), r.to(DEV), h0.to(DEV), cu.to(DEV), picard_iters=P,
                               eps=EPS)
    for s in range(len(lengths)):
        a, b = int(cu[s]), int(cu[s + 1])
        want = _walk(wx[:, a:b].double(), r.double(), h0[s:s + 1].double(), P)
        _check(got[:, a:b], want, b - a, P)


@pytest.mark.parametrize("lengths", [[4096] + [17] * 40, [2500, 31, 900, 700, 12, 60], None])
def test_repeats_bit_for_bit(lengths):
    """float32 warm starts do not depend on the order in which tiles finish."""
    d, B, N = (64, 1, sum(lengths)) if lengths else (200, 3, 4097)
    g = torch.Generator().manual_seed(N)
    wx = torch.randn(B, N, 4 * d, generator=g).to(DEV)
    r = (torch.randn(4, d, generator=g) * 0.3).to(DEV)
    h0 = torch.rand(len(lengths) if lengths else B, 4, d, generator=g).to(DEV)
    cu = torch.tensor([0, *torch.tensor(lengths).cumsum(0).tolist()]).to(DEV) if lengths else None
    print(f"case repeats B={B} N={N} packed={lengths is not None}", flush=True)
    outs = [ops.slstm_init_fused(wx, r, h0, cu, picard_iters=3, eps=EPS) for _ in range(30)]
    prev = torch.are_deterministic_algorithms_enabled()
    torch.use_deterministic_algorithms(True, warn_only=True)
    try:
        outs.append(ops.slstm_init_fused(wx, r, h0, cu, picard_iters=3, eps=EPS))
    finally:
        torch.use_deterministic_algorithms(prev)
    assert all(torch.equal(o, outs[0]) for o in outs[1:])
