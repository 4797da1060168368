"""Head GRU as walks over time (one per sequence and head) at the edges of its
16-step blocks, against the oracle, the oracle's float64 gradients and the
chunked scan; and the routing between the two.

fp32 bars: 1e-5 absolute forward (states in (-1, 1)), 1e-5 of the largest entry
for the gradients.  The chunked scan's backward, linear in its chunk transfers,
is off by up to 2^-9 (their bf16 operands) of what crosses a chunk of 32 steps;
under these weights (spectral norm ~3) that share stays below 1%: 2e-5."""

import pytest
import torch

import oracle as O
from oracle.backward import gru_head_backward
from oracle.ragged import gru_head_newton_ragged

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.fixture(params=["walk", "chunked"])
def route(request, monkeypatch):
    monkeypatch.setenv("PARARNN_AMD_GRU_WALK", "1" if request.param == "walk" else "0")
    monkeypatch.setenv("PARARNN_AMD_CHECK_STATUS", "1")
    return request.param


def _params(H, dh, seed, scale=0.2):
    g = torch.Generator().manual_seed(seed)
    d = H * dh
    return O.GRUHeadParams(torch.randn(3 * d, 8, generator=g) * 0.3,
                           torch.randn(3 * d, generator=g) * 0.1,
                           *(torch.randn(H, dh, dh, generator=g) * scale for _ in range(3)))


def _mats(p, dtype=torch.float32):
    return [a.to(DEV, dtype) for a in p.mats()]


@pytest.mark.parametrize("T", [1, 15, 16, 17, 31, 32, 33, 48, 49, 200])
@pytest.mark.parametrize("K", [1, 2, 4])
@pytest.mark.parametrize("with_h0", [False, True])
def test_forward_vs_oracle(T, K, with_h0, route):
    from pararnn_amd import ops

    print(f"case forward T={T} K={K} h0={with_h0} {route}", flush=True)
    B, H = (3, 2) if T < 50 else (2, 1)
    p = _params(H, 64, T + K)
    x = torch.randn(B, T, 8, generator=torch.Generator().manual_seed(T))
    h0 = torch.rand(B, 64 * H, generator=torch.Generator().manual_seed(1)) - 0.5 \
        if with_h0 else None
    wx = p.wx(x)
    out = ops.newton_gru_head_fused(wx.to(DEV), *_mats(p), None if h0 is None else h0.to(DEV),
                                    max_iters=K, omega=0.9).cpu()
    ref = O.gru_head_newton(p, x, max_iters=K, h0=h0, omega=0.9)
    err = (out - ref).abs().max().item()
    print(f"  max|gpu - oracle| {err:.2e}", flush=True)
    assert err <= 1e-5


@pytest.mark.parametrize("T", [1, 15, 16, 17, 33, 64, 130])
@pytest.mark.parametrize("with_h0", [False, True])
def test_backward_vs_float64(T, with_h0, route):
    from pararnn_amd import ops

    print(f"case backward T={T} h0={with_h0} {route}", flush=True)
    B, H = 2, 2
    p = _params(H, 64, T)
    g = torch.Generator().manual_seed(T + 9)
    x = torch.randn(B, T, 8, generator=g)
    st = torch.tanh(torch.randn(B, T, 64 * H, generator=g))
    gr = torch.randn(B, T, 64 * H, generator=g)
    h0 = torch.rand(B, 64 * H, generator=g) - 0.5 if with_h0 else None
    wx = p.wx(x)
    g_wx, g_a, g_h0 = ops.gru_head_backward_fused(
        wx.to(DEV), *_mats(p), None if h0 is None else h0.to(DEV), st.to(DEV), gr.to(DEV))
    p64 = O.GRUHeadParams(*(v.double() for v in (p.W, p.b, p.A_z, p.A_r, p.A_n)))
    ref = gru_head_backward(p64, x.double(), st.double(), gr.double(),
                            h0=None if h0 is None else h0.double(), wx=wx.double())
    pairs = [("g_wx", g_wx, ref["g_wx"])] + [(k, g_a[i], ref[k]) for i, k in
                                             enumerate(("A_z", "A_r", "A_n"))]
    if with_h0:
        pairs.append(("h0", g_h0, ref["h0"]))
    for k, a, b in pairs:
        e = ((a.cpu().double() - b).abs().max() / b.abs().max().clamp_min(1e-30)).item()
        print(f"  {k} rel {e:.2e}", flush=True)
        assert e <= (1e-5 if route == "walk" else 2e-5), k


@pytest.mark.parametrize("lengths", [[1], [16, 1, 17, 15, 33], [1] * 20, [100] + [3] * 30])
@pytest.mark.parametrize("with_h0", [False, True])
def test_packed_vs_each_sequence(lengths, with_h0, route):
    from pararnn_amd import ops

    print(f"case packed {lengths[:6]} h0={with_h0} {route}", flush=True)
    H, N, S = 2, sum(lengths), len(lengths)
    p = _params(H, 64, N)
    g = torch.Generator().manual_seed(N)
    x = torch.randn(1, N, 8, generator=g)
    h0 = torch.rand(S, 64 * H, generator=g) - 0.5 if with_h0 else None
    cs = torch.tensor([0] + lengths).cumsum(0)
    wx, mats = p.wx(x).to(DEV), _mats(p)
    hd = None if h0 is None else h0.to(DEV)
    out = ops.newton_gru_head_fused(wx, *mats, hd, cs.to(DEV), max_iters=3, omega=1.0)
    ref = gru_head_newton_ragged(p, x, cs, max_iters=3, h0=h0)
    assert (out.cpu() - ref).abs().max().item() <= 1e-5
    gr = torch.randn(1, N, 64 * H, generator=g).to(DEV)
    g_wx, g_a, g_h0 = ops.gru_head_backward_fused(wx, *mats, hd, out, gr, cs.to(DEV))
    acc = torch.zeros_like(g_a)
    for s in range(S):
        a, b = int(cs[s]), int(cs[s + 1])
        r = ops.gru_head_backward_fused(wx[:, a:b], *mats, None if hd is None else hd[s:s + 1],
                                        out[:, a:b], gr[:, a:b])
        bar = 1e-5 if route == "walk" else 2e-5
        assert (g_wx[:, a:b] - r[0]).abs().max() <= bar * r[0].abs().max().clamp_min(1e-3)
        if with_h0:
            assert (g_h0[s] - r[2][0]).abs().max() <= bar * r[2].abs().max().clamp_min(1e-3)
        acc += r[1]
    assert (g_a - acc).abs().max() <= bar * acc.abs().max()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("T", [17, 100])
def test_16_bit_storage_matches_the_chunked_scan(dtype, T, monkeypatch):
    """The same fp32 work on 16-bit operands: the routes differ by the last
    stored bit of a value (u = 2^-8 / 2^-11 of it), and dL/dA, a sum of products
    of such values, by u in the 2-norm at most."""
    from pararnn_amd import ops

    print(f"case 16 bit {dtype} T={T}", flush=True)
    H, B = 2, 3
    p = _params(H, 64, T)
    g = torch.Generator().manual_seed(T)
    wx = p.wx(torch.randn(B, T, 8, generator=g)).to(DEV, dtype)
    h0 = (torch.rand(B, 64 * H, generator=g) - 0.5).to(DEV, dtype)
    gr = torch.randn(B, T, 64 * H, generator=g).to(DEV, dtype)
    res = {}
    for v in "01":
        monkeypatch.setenv("PARARNN_AMD_GRU_WALK", v)
        out = ops.newton_gru_head_fused(wx, *_mats(p, dtype), h0, max_iters=3, omega=1.0)
        res[v] = [out, *ops.gru_head_backward_fused(wx, *_mats(p, dtype), h0,
                                                    res["0"][0] if v == "1" else out, gr)]
    u = 2.0 ** (-8 if dtype is torch.bfloat16 else -11)
    for a, b in zip(res["1"], res["0"]):
        assert (a.float() - b.float()).norm() <= u * b.float().norm()


def test_more_walks_than_fit_at_once(monkeypatch):
    """1200 workgroups per iteration: later ones start when earlier ones end."""
    from pararnn_amd import ops

    monkeypatch.setenv("PARARNN_AMD_GRU_WALK", "1")
    monkeypatch.setenv("PARARNN_AMD_CHECK_STATUS", "1")
    print("case 1200 walks per iteration", flush=True)
    B, T, H = 400, 37, 3
    p = _params(H, 64, 5)
    wx = p.wx(torch.randn(B, T, 8, generator=torch.Generator().manual_seed(2))).to(DEV)
    out = ops.newton_gru_head_fused(wx, *_mats(p), max_iters=3, omega=1.0)
    monkeypatch.setenv("PARARNN_AMD_GRU_WALK", "0")
    ref = ops.newton_gru_head_fused(wx, *_mats(p), max_iters=3, omega=1.0)
    assert (out - ref).abs().max().item() <= 1e-5


def test_graph_replays(monkeypatch):
    """Captured once and replayed with eager calls between: each replay equals the eager result
    on the inputs it finds."""
    from pararnn_amd import ops

    monkeypatch.setenv("PARARNN_AMD_GRU_WALK", "1")
    print("case graph replays", flush=True)
    p = _params(2, 64, 3)
    mats = _mats(p)
    g = torch.Generator().manual_seed(4)
    xs = [p.wx(torch.randn(3, 50, 8, generator=g)).to(DEV) for _ in range(4)]
    wx = xs[0].clone()
    gr = torch.randn(3, 50, 128, generator=g).to(DEV)

    def call(w):
        out = ops.newton_gru_head_fused(w, *mats, max_iters=3, omega=1.0)
        return [out, *ops.gru_head_backward_fused(w, *mats, None, out, gr)[:2]]

    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        call(wx)
    torch.cuda.current_stream().wait_stream(side)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        held = call(wx)
    for x in xs:
        want = call(x)
        wx.copy_(x)
        graph.replay()
        torch.cuda.synchronize()
        for a, b in zip(held, want):
            assert torch.equal(a, b)


@pytest.mark.parametrize("walk", ["0", "1", None])
def test_packed_call_with_int32_offsets_is_captured(walk, monkeypatch):
    """Known int32 offsets: a repeated packed call reads nothing back, so it can be
    captured; each replay equals the eager result."""
    from pararnn_amd import ops

    if walk is None:
        monkeypatch.delenv("PARARNN_AMD_GRU_WALK", raising=False)
    else:
        monkeypatch.setenv("PARARNN_AMD_GRU_WALK", walk)
    print(f"case packed int32 capture walk={walk}", flush=True)
    p = _params(2, 64, 3)
    mats = _mats(p)
    g = torch.Generator().manual_seed(5)
    cs = torch.tensor([0, 17, 33, 34, 90], dtype=torch.int32, device=DEV)
    xs = [p.wx(torch.randn(1, 90, 8, generator=g)).to(DEV) for _ in range(3)]
    wx = xs[0].clone()
    h0 = (torch.rand(4, 128, generator=g) - 0.5).to(DEV)
    gr = torch.randn(1, 90, 128, generator=g).to(DEV)

    def call(w):
        out = ops.newton_gru_head_fused(w, *mats, h0, cs, max_iters=3, omega=1.0)
        return [out, *ops.gru_head_backward_fused(w, *mats, h0, out, gr, cs)]

    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        call(wx)
    torch.cuda.current_stream().wait_stream(side)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        held = call(wx)
    for x in xs:
        want = call(x)
        wx.copy_(x)
        graph.replay()
        torch.cuda.synchronize()
        for a, b in zip(held, want):
            assert torch.equal(a, b)


def test_two_streams(monkeypatch):
    """Solves of two streams at once keep apart (a workspace each)."""
    from pararnn_amd import ops

    monkeypatch.setenv("PARARNN_AMD_GRU_WALK", "1")
    print("case two streams", flush=True)
    p = _params(2, 64, 6)
    mats = _mats(p)
    g = torch.Generator().manual_seed(7)
    xs = [p.wx(torch.randn(4, 300, 8, generator=g)).to(DEV) for _ in range(2)]
    want = [ops.newton_gru_head_fused(x, *mats, max_iters=3, omega=1.0) for x in xs]
    streams = [torch.cuda.Stream() for _ in xs]
    torch.cuda.synchronize()
    got = [[], []]
    for _ in range(5):
        for i, s in enumerate(streams):
            with torch.cuda.stream(s):
                got[i].append(ops.newton_gru_head_fused(xs[i], *mats, max_iters=3, omega=1.0))
    torch.cuda.synchronize()
    for i in range(2):
        for o in got[i]:
            assert torch.equal(o, want[i])


@pytest.mark.parametrize("room", ["kept", "own", "none"])
def test_each_workspace_gives_the_same_states(room, monkeypatch):
    """From the stream's cache, from a buffer of the call's own (other values in it), and
    with no room for either (the chunked scan, at its own bar); nothing of a buffer of
    the call's own stays."""
    from pararnn_amd import ops

    monkeypatch.setenv("PARARNN_AMD_GRU_WALK", "1")
    monkeypatch.setenv("PARARNN_AMD_CHECK_STATUS", "1")
    print(f"case workspace {room}", flush=True)
    p = _params(3, 64, 9)
    wx = p.wx(torch.randn(4, 300, 8, generator=torch.Generator().manual_seed(9))).to(DEV)
    want = ops.newton_gru_head_fused(wx, *_mats(p), max_iters=3, omega=1.0)
    ops.release_workspaces()
    if room != "kept":
        monkeypatch.setattr(ops, "_WALK_KEEP", 0)
    if room == "none":
        monkeypatch.setattr(ops, "_wide_workspace_cap", lambda d: 0)
    torch.full((1 << 24,), float("nan"), device=DEV)  # what a fresh buffer may hold
    for _ in range(2):
        got = ops.newton_gru_head_fused(wx, *_mats(p), max_iters=3, omega=1.0)
        if room == "none":
            assert (got - want).abs().max().item() <= 1e-5
        else:
            assert torch.equal(got, want)
    assert bool(ops._tagged) is (room == "kept")


def test_threads_on_one_stream(monkeypatch):
    """Four threads on the default stream, each with solves of its own."""
    import threading

    from pararnn_amd import ops

    monkeypatch.setenv("PARARNN_AMD_GRU_WALK", "1")
    print("case four threads, one stream", flush=True)
    p = _params(2, 64, 6)
    mats = _mats(p)
    g = torch.Generator().manual_seed(8)
    xs = [p.wx(torch.randn(2 + i, 200, 8, generator=g)).to(DEV) for i in range(4)]
    want = [ops.newton_gru_head_fused(x, *mats, max_iters=3, omega=1.0) for x in xs]
    got = [[] for _ in xs]

    def work(i):
        for _ in range(10):
            got[i].append(ops.newton_gru_head_fused(xs[i], *mats, max_iters=3, omega=1.0))

    threads = [threading.Thread(target=work, args=(i,)) for i in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    torch.cuda.synchronize()
    for w, outs in zip(want, got):
        assert len(outs) == 10 and all(torch.equal(o, w) for o in outs)
