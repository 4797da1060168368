"""The gate split of the sLSTM Newton kernels at and next to ties.

One Newton iteration on steps whose left = z_f + m and z_i are equal (the max's
derivative is split 0.5 / 0.5), one float apart, 1e-30 apart, or up
to 60 apart (the smaller gate, e^-60, is nothing beside the larger), in fp32, against the cell's own step and Jacobian in float64: an
iteration is H + delta with delta_t = J_t delta_{t-1} + F_t, so with T = 2 steps the
second one shows J.  Tolerance: 40 operations of relative error 2^-23 on terms
of at most 8 in size (each derivative is at most 4, delta at most 2)."""

import pytest
import torch

from pararnn_amd import ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("gap", [0.0, 1.2e-7, -1.2e-7, 1e-30, -1e-30, 0.5, -3.0, 60.0, -60.0])
def test_one_iteration_next_to_a_tie(gap):
    d = 70
    g = torch.Generator().manual_seed(3)
    wx = torch.randn(1, 2, 4, d, generator=g, dtype=torch.float64) * 0.5
    guess = torch.rand(1, 2, 4, d, generator=g, dtype=torch.float64) * 0.5 + 0.5
    r = torch.randn(4, d, generator=g, dtype=torch.float64) * 0.3
    r[:2] = 0.0  # the gates' difference is then exactly z_f + m - z_i
    guess[:, 0, 2] = 0.0
    wx[:, 1, 1] = gap
    wx[:, 1, 0] = 0.0
    wx, guess, r = (t.float() for t in (wx, guess, r))
    out = ops.newton_slstm_fused(wx.reshape(1, 2, 4 * d).cuda(), r.cuda(), None, guess.cuda(),
                                 max_iters=1, omega=1.0, eps=1e-6).double().cpu()
    x, h, R = wx.double(), guess.double(), r.double()

    def step(prev, t):
        z = x[0, t] + R * prev[3]
        left = z[1] + prev[2]
        m = torch.maximum(left, z[0])
        f, i = torch.exp(left - m), torch.exp(z[0] - m)
        n = f * prev[1] + i
        c = f * prev[0] + i * torch.tanh(z[2])
        return torch.stack([c, n, m, torch.sigmoid(z[3]) * c / (n + 1e-6)])

    d0 = step(torch.zeros(4, d, dtype=torch.float64), 0) - h[0, 0]
    pred, jv = torch.autograd.functional.jvp(lambda p: step(p, 1), h[0, 0], d0)
    want = torch.stack([h[0, 0] + d0, jv + pred])
    assert (out[0] - want).abs().max().item() <= 40 * 2.0 ** -23 * 8
