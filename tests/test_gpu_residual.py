"""The residual kernels against the cells' own tensor ops.

Both evaluate f(H_{t-1}, x_t) with the same rounding points, so a difference
of one element differs by the last bits of its terms: with u the unit roundoff
of the storage type (float32 arithmetic below it), |f - H| moves by at most a
few u of |f| + |H|.  The bars take 8 u of the largest |f| + |H| (float32: the
recurrent products are 128-term sums in another order, 128 u / 2 more)."""

import pytest
import torch

from pararnn_amd import NewtonConfig, NewtonStats, ParaGRU, ParaSLSTM, newton_apply, ops
from pararnn_amd.newton import _max_residual, _prepend_any

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
UNIT = {torch.float32: 2.0 ** -24, torch.bfloat16: 2.0 ** -9, torch.float16: 2.0 ** -12}


def _reference(cell, wx, states, h0, cu):
    with torch.no_grad():
        pred = cell.step(_prepend_any(states, h0, cu), None, wx=wx)
        return float((pred - states).abs().amax()), float((pred.abs() + states.abs()).amax())


def _offsets(n, seqs):
    return torch.tensor([round(i * n / seqs) for i in range(seqs + 1)], device=DEV)


@pytest.mark.parametrize("dtype", list(UNIT))
@pytest.mark.parametrize("B,T,d,seqs", [(1, 1, 1, 0), (2, 8, 63, 0), (3, 17, 64, 0),
                                        (2, 33, 65, 0), (2, 500, 200, 0), (1, 95, 70, 7),
                                        (1, 40, 64, 40)])
@pytest.mark.parametrize("with_h0", [False, True])
def test_slstm_matches_tensor_ops(dtype, B, T, d, seqs, with_h0):
    torch.manual_seed(B * 100 + T + d)
    cell = ParaSLSTM(8, d, device=DEV).to(dtype)
    wx = torch.randn(B, T, 4 * d, device=DEV).to(dtype)
    rows = seqs or B
    n = torch.rand(B, T, 1, d, device=DEV) * 5 + 0.5
    states = torch.cat([n * 0.3, n, torch.randn(B, T, 2, d, device=DEV)], 2).to(dtype)
    h0 = torch.rand(rows, 4, d, device=DEV).to(dtype) if with_h0 else None
    cu = _offsets(T, seqs) if seqs else None
    want, scale = _reference(cell, wx, states, h0, cu)
    got = _max_residual(cell, wx, states, h0, cu)
    print(f"  {dtype} {B}x{T}x{d} seqs={seqs}: kernel {got:.6g} tensor ops {want:.6g}", flush=True)
    assert abs(got - want) <= 8 * UNIT[dtype] * scale


@pytest.mark.parametrize("dtype", list(UNIT))
@pytest.mark.parametrize("B,T,H,dh,seqs", [(1, 1, 1, 1, 0), (2, 31, 3, 16, 0), (1, 32, 5, 24, 0),
                                           (2, 33, 2, 64, 0), (3, 200, 2, 65, 0),
                                           (1, 70, 3, 128, 0), (1, 97, 4, 48, 9),
                                           (1, 64, 2, 128, 64)])
@pytest.mark.parametrize("with_h0", [False, True])
def test_gru_matches_tensor_ops(dtype, B, T, H, dh, seqs, with_h0):
    torch.manual_seed(B * 100 + T + dh)
    d = H * dh
    cell = ParaGRU(8, d, mix="head", n_heads=H).to(DEV).to(dtype)
    wx = torch.randn(B, T, 3 * d, device=DEV).to(dtype)
    states = torch.tanh(torch.randn(B, T, d, device=DEV)).to(dtype)
    h0 = torch.tanh(torch.randn(seqs or B, d, device=DEV)).to(dtype) if with_h0 else None
    cu = _offsets(T, seqs) if seqs else None
    want, scale = _reference(cell, wx, states, h0, cu)
    got = _max_residual(cell, wx, states, h0, cu)
    print(f"  {dtype} {B}x{T} H={H} dh={dh} seqs={seqs}: kernel {got:.6g} tensor ops {want:.6g}",
          flush=True)
    assert abs(got - want) <= (72 if dtype is torch.float32 else 8) * UNIT[dtype] * scale


@pytest.mark.parametrize("kind", ["slstm", "gru"])
def test_one_bad_value_anywhere_is_seen(kind):
    """NaN wins over every finite difference and infinity over every number, as in amax."""
    torch.manual_seed(0)
    d, T = 130, 77
    cell = ParaSLSTM(4, d, device=DEV) if kind == "slstm" else \
        ParaGRU(4, d, mix="head", n_heads=2).to(DEV)
    wx = torch.randn(1, T, (4 if kind == "slstm" else 3) * d, device=DEV)
    shape = (1, T, 4, d) if kind == "slstm" else (1, T, d)
    for t in (0, 40, T - 1):
        for bad in (float("nan"), float("inf")):
            states = torch.rand(*shape, device=DEV)
            states[0, t, ..., d - 1] = bad
            want, _ = _reference(cell, wx, states, None, None)
            got = _max_residual(cell, wx, states, None, None)
            assert str(got) == str(want), (t, bad, got, want)


def test_own_step_of_a_subclass_is_evaluated():
    class Shifted(ParaSLSTM):
        def step(self, state_prev, x=None, *, wx=None):
            return super().step(state_prev, x, wx=wx) + 1.0

    torch.manual_seed(0)
    cell = Shifted(8, 16, device=DEV)
    x = torch.randn(2, 20, 8, device=DEV) * 0.5
    st = NewtonStats()
    with torch.no_grad():
        newton_apply(cell, x, NewtonConfig(residual_fail=None, picard_adapt=False), stats=st)
    assert abs(st.max_residual - 1.0) < 1e-3


@pytest.mark.parametrize("config", [{}, {"scan_backend": "eager", "residual_atol": None},
                                    {"chunk_len": 8, "picard_adapt": False}])
def test_step_without_wx_passes_the_default_gate(config):
    """A step of two arguments that agrees with the library's: the gate accepts the solve."""
    class Two(ParaSLSTM):
        def step(self, state_prev, x):
            return super().step(state_prev, x)

    torch.manual_seed(0)
    cell = Two(8, 16, device=DEV)
    x = torch.randn(2, 20, 8, device=DEV) * 0.5
    st = NewtonStats()
    with torch.no_grad():
        newton_apply(cell, x, NewtonConfig(**config), stats=st)
    assert st.max_residual < 1e-3


def test_residual_rejects_mismatched_operands():
    wx = torch.zeros(1, 4, 12, device=DEV)
    a = torch.zeros(1, 4, 4, device=DEV)
    with pytest.raises(ValueError):
        ops.gru_head_residual(wx, a, a, a, None, torch.zeros(1, 3, 4, device=DEV))
    with pytest.raises(TypeError):
        ops.gru_head_residual(torch.zeros(1, 4, 387, device=DEV), *(
            torch.zeros(1, 129, 129, device=DEV),) * 3, None, torch.zeros(1, 4, 129, device=DEV))
    with pytest.raises(ValueError):
        ops.slstm_residual(torch.zeros(1, 4, 16, device=DEV), torch.zeros(4, 4, device=DEV),
                           torch.zeros(2, 4, 4, device=DEV), torch.zeros(1, 4, 4, 4, device=DEV),
                           eps=1e-6)
