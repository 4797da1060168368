"""The residual of cells whose step is not the library's own, on the CPU: it is what
that step says, from the cell's input, whatever other arguments the step has."""

import pytest
import torch

from pararnn_amd import NewtonConfig, NewtonStats, ParaGRU, ParaSLSTM
from pararnn_amd.newton import _fill_stats


class _TwoArgs(ParaSLSTM):
    def step(self, state_prev, x):
        return super().step(state_prev, x) + 0.25


class _Reads(ParaGRU):
    def step(self, h_prev, x=None, *, wx=None):
        return super().step(h_prev, x, wx=wx) + x.mean()


def _patched(prev, x):
    return prev * 0.0 + 3.0


@pytest.mark.parametrize("packed", [False, True])
@pytest.mark.parametrize("wx_at_hand", [False, True])
@pytest.mark.parametrize("kind", ["two_args", "reads_x", "instance"])
def test_own_steps_get_the_input(kind, wx_at_hand, packed):
    torch.manual_seed(1)
    if kind == "reads_x":
        cell = _Reads(8, 8, mix="head", n_heads=2)
    else:
        cell = (_TwoArgs if kind == "two_args" else ParaSLSTM)(8, 8)
        if kind == "instance":
            cell.step = _patched
    tail = (8,) if kind == "reads_x" else (4, 8)
    x = torch.randn(1, 6, 8)
    states = torch.rand(1, 6, *tail) + 0.5
    cu = torch.tensor([0, 2, 6]) if packed else None
    h0 = torch.rand(2 if packed else 1, *tail)
    prev = torch.cat([h0[:1, None], states[:, :-1]], 1)
    if packed:
        prev[:, 2] = h0[1]
    stats = NewtonStats()
    with torch.no_grad():
        want = (cell.step(prev, x) - states).abs().max().item()
        _fill_stats(cell, x, states, h0, NewtonConfig(residual_fail=None, picard_adapt=False),
                    iters=3, stats=stats, cu_seqlens=cu, wx=cell.W_x(x) if wx_at_hand else None)
    assert stats.max_residual == want
