"""decode_step from the cell's input: the projection in the step's kernel.

Inputs whose projection is exact in every order of summation and in the storage
type (small multiples of 2^-2, |wx| 2^4 <= 256), so the step from x equals the step
from the GEMM's wx bit for bit: partly filled tiles of rows and channels, d_in of
one load, of a partial and of more than one turn, in place and through a block table."""

import pytest
import torch

from pararnn_amd import decode as D
from pararnn_amd.cells import ParaGRU, ParaSLSTM

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _case(kind, B, d, d_in, dtype, bias=True):
    g = torch.Generator().manual_seed(B * 10000 + d * 10 + d_in)
    if kind == "slstm":
        cell = ParaSLSTM(d_in, d)
    else:
        cell = ParaGRU(d_in, d, mix="diag") if kind == "diag" else \
            ParaGRU(d_in, d, mix="head", n_heads=d // 64)
    cell = cell.to(DEV, dtype)

    def q(*shape):  # -1/4, 0, 1/4
        return (torch.randint(-1, 2, shape, generator=g) / 4).to(DEV, dtype)

    with torch.no_grad():
        cell.W_x.weight.copy_(q(*cell.W_x.weight.shape))
        cell.W_x.bias.copy_(q(*cell.W_x.bias.shape))
    if not bias:
        cell.W_x.bias = None
    x = q(B, d_in)
    wx = torch.nn.functional.linear(x.float(), cell.W_x.weight.float())
    assert wx.abs().max().item() * 16 <= 252
    state = torch.rand(B, 4, d, generator=g) if kind == "slstm" else torch.rand(B, d, generator=g)
    return cell, x, state.to(DEV, dtype)


SHAPES = [("slstm", 1, 5, 8), ("slstm", 16, 64, 64), ("slstm", 17, 63, 136), ("slstm", 33, 300, 40),
          ("slstm", 64, 130, 1032), ("slstm", 65, 1024, 136), ("slstm", 130, 516, 128),
          ("slstm", 3, 2048, 1024), ("diag", 1, 1, 16), ("diag", 31, 66, 72), ("diag", 70, 600, 24),
          ("head", 1, 64, 64), ("head", 9, 128, 520), ("head", 67, 192, 72)]


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("kind,B,d,d_in", SHAPES)
def test_step_from_x_equals_step_from_wx(kind, B, d, d_in, dtype, monkeypatch):
    monkeypatch.setattr(D, "_small_step", lambda *a: True)
    took = []
    launch = D._launch
    monkeypatch.setattr(D, "_launch", lambda *a: (took.append(a[5]), launch(*a))[1])
    cell, x, state = _case(kind, B, d, d_in, dtype, bias=d % 2 == 0)
    with torch.no_grad():
        wx = cell.W_x(x)
        want = D.decode_step(cell, state, wx=wx)
        got = D.decode_step(cell, state, x)
        assert took[0] is None and took[1] is cell.W_x
        assert torch.equal(got, want)
        # in place, through a pool in another order
        pool = torch.randn(B + 3, *state.shape[1:], device=DEV, dtype=dtype)
        table = torch.randperm(B + 3, generator=torch.Generator().manual_seed(1))[:B].to(DEV)
        pool[table] = state
        ref = pool.clone()
        ref[table] = want
        D.decode_step(cell, pool, x[:, None], block_table=table.int())
        assert took[-1] is cell.W_x and torch.equal(pool, ref)


def test_captured_replays_and_an_input_that_is_the_state():
    """Replays equal live steps; a GRU fed its own state in place takes the
    library projection (the kernel would overwrite rows it still reads)."""
    cell, x, state = _case("diag", 8, 64, 64, torch.float32)
    out = torch.empty_like(state)
    with torch.no_grad():
        want = D.decode_step(cell, state, x)
        side = torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            D.decode_step(cell, state, x, out=out)
        torch.cuda.current_stream().wait_stream(side)
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            D.decode_step(cell, state, x, out=out)
        for _ in range(3):
            out.fill_(-1.0)
            graph.replay()
            torch.cuda.synchronize()
            assert torch.equal(out, want)
        ref = D.decode_step(cell, state, wx=cell.W_x(state))
        own = state.clone()
        D.decode_step(cell, own, own, out=own)
        assert torch.equal(own, ref)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_route_at_the_line(dtype, monkeypatch):
    """The rule as it stands, on either side of its line: one row below it (and on it)
    the kernel projects, one row above it the library; same step."""
    d_in = 1024
    rows = (1 << (26 if dtype is torch.bfloat16 else 24)) // (d_in * d_in)
    took = []
    launch = D._launch
    monkeypatch.setattr(D, "_launch", lambda *a: (took.append(a[5]), launch(*a))[1])
    for B, projects in ((rows - 1, True), (rows, True), (rows + 1, False)):
        g = torch.Generator().manual_seed(B)
        cell = ParaSLSTM(d_in, d_in).to(DEV, dtype)
        with torch.no_grad():
            w = torch.zeros(4 * d_in, d_in)
            w[:, :32] = torch.randint(-1, 2, (4 * d_in, 32), generator=g) / 4
            cell.W_x.weight.copy_(w)
            x = (torch.randint(-1, 2, (B, d_in), generator=g) / 4).to(DEV, dtype)
            state = torch.rand(B, 4, d_in, generator=g).to(DEV, dtype)
            want = D.decode_step(cell, state, wx=cell.W_x(x))
            got = D.decode_step(cell, state, x)
        assert (took[-1] is cell.W_x) is projects
        assert torch.equal(got, want)
