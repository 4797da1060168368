"""Which head-GRU calls run as walks over time and which as the chunked scan
(``ops._walks``), on the CPU."""

import pytest

from pararnn_amd import ops


@pytest.fixture(autouse=True)
def _plain(monkeypatch):
    for k in ("PARARNN_AMD_GRU_WALK", *ops._CHUNK_SWITCHES):
        monkeypatch.delenv(k, raising=False)


@pytest.mark.parametrize("units,T,iters,walk", [
    (1, 33, 3, True), (1, 128, 0, True), (8, 128, 3, True), (128, 1024, 3, True),
    (512, 3000, 1, True), (512, 1024, 0, True), (32, 3000, 3, True),
    (1, 8192, 3, False), (8, 4096, 3, False), (32, 8192, 3, False), (32, 32768, 3, False),
    (64, 1024, 1, False), (64, 3000, 0, False), (1, 1024, 1, False)])
def test_rectangular(units, T, iters, walk):
    assert ops._walks(units, units * T, T, iters) is walk


def test_one_long_sequence_among_short_ones_stays_chunked():
    assert not ops._walks(64 * 8, (65536 + 63 * 1024) * 8, 65536, 3)
    assert ops._walks(64 * 8, 64 * 1024 * 8, 1024, 3)


def test_switches(monkeypatch):
    assert not ops._walks(128, 128 * 128, 128, ops._WALK_MAX_ITERS + 1)
    monkeypatch.setenv("PRNN_GRU_REPLAY_MFMA", "1")
    assert not ops._walks(128, 128 * 128, 128, 3)
    monkeypatch.setenv("PARARNN_AMD_GRU_WALK", "1")
    assert ops._walks(1, 10**6, 10**6, 3)
    assert not ops._walks(1, 16, 16, ops._WALK_MAX_ITERS + 1)
    monkeypatch.setenv("PARARNN_AMD_GRU_WALK", "0")
    assert not ops._walks(128, 128 * 128, 128, 3)


def test_longest_sequence_follows_the_offsets():
    import torch

    from pararnn_amd.ragged import longest_sequence, validate_cu_seqlens

    cs = torch.tensor([0, 3, 10, 12])
    assert longest_sequence(validate_cu_seqlens(cs, 12), 12) == 7
    cs[1] = 9
    assert longest_sequence(validate_cu_seqlens(cs, 12), 12) == 9
    other = torch.tensor([0, 5, 12])
    assert longest_sequence(other, 12) == 7


def test_walk_workspaces_kept_are_bounded(monkeypatch):
    """Small ones come from the stream's cache, larger ones belong to the call (tag 0: it
    clears them), and what is over the cap or not to be had sends the call to the scan."""
    import torch

    dev = torch.device("cuda", 0)
    full = []

    def temporary(n, d):
        if full:
            raise torch.OutOfMemoryError("no room")
        return "own"

    monkeypatch.setattr(ops, "_wide_workspace_cap", lambda d: 1 << 33)
    monkeypatch.setattr(ops, "_workspace", temporary)
    monkeypatch.setattr(ops, "_slstm_workspace", lambda n, d, k: (temporary(n, d) and "kept", 65))
    keep = ops._WALK_KEEP
    assert keep <= 1 << 30
    assert ops._walk_workspace(keep, dev, (0, 0)) == ("kept", 65)
    assert ops._walk_workspace(keep + 1, dev, (0, 0)) == ("own", 0)
    assert ops._walk_workspace((1 << 33) + 1, dev, (0, 0)) is None
    full.append(1)
    assert ops._walk_workspace(keep, dev, (0, 0)) is None
    assert ops._walk_workspace(keep + 1, dev, (0, 0)) is None


def test_a_growing_cache_gives_its_buffer_back_first(monkeypatch):
    import gc
    import weakref

    import torch

    class _S:
        cuda_stream = 77

    alive = []
    real = torch.zeros

    def zeros(n, dtype, device):
        gc.collect()
        alive.append([r() is not None for r in made])
        out = real(n, dtype=dtype)
        made.append(weakref.ref(out))
        return out

    made = []
    monkeypatch.setattr(ops.torch, "zeros", zeros)
    monkeypatch.setattr(ops.torch.cuda, "is_current_stream_capturing", lambda: False)
    monkeypatch.setattr(ops.torch.cuda, "current_stream", lambda d: _S)
    ops.release_workspaces()
    dev = torch.device("cuda", 0)
    for n in (1024, 4096, 65536):
        ops._slstm_workspace(n, dev)
    assert alive == [[], [False], [False, False]]
    ops.release_workspaces()


def test_threads_on_one_stream_take_turns(monkeypatch):
    """From picking the tag to the launch (buffers on the CPU, a library that only looks):
    two calls at once would clear one buffer's tickets twice and then launch twice."""
    import contextlib
    import threading
    import time

    import torch

    inside, seen, wrong = [], [], []

    class _Lib:
        def prnn_gru_head_walk_newton_workspace_size(self, *a):
            return 4096

        def prnn_gru_head_walk_newton(self, *a):
            tag = a[-2]
            if inside:
                wrong.append(("together", tag))
            inside.append(tag)
            time.sleep(0.02)
            seen.append(tag)
            inside.pop()
            return 0

    class _S:
        cuda_stream = 0

    monkeypatch.setattr(ops._lib, "load", _Lib)
    monkeypatch.setattr(ops._lib, "check", lambda rc, what: None)
    monkeypatch.setattr(ops, "_validate", lambda *a: 0)
    monkeypatch.setattr(ops, "_stream", lambda d: 0)
    monkeypatch.setattr(ops, "_walks", lambda *a: True)
    monkeypatch.setattr(ops, "_wide_workspace_cap", lambda d: 1 << 30)
    monkeypatch.setattr(ops.torch.cuda, "device", lambda d: contextlib.nullcontext())
    monkeypatch.setattr(ops.torch.cuda, "current_device", lambda: 0)
    monkeypatch.setattr(ops.torch.cuda, "current_stream", lambda d: _S)
    monkeypatch.setattr(ops.torch.cuda, "is_current_stream_capturing", lambda: False)
    ops.release_workspaces()
    a = torch.zeros(1, 64, 64)
    wx = torch.zeros(1, 3, 192)

    def work():
        for _ in range(5):
            ops._gru_head_dense(wx, a, a, a, None, 3, 1.0)

    threads = [threading.Thread(target=work) for _ in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    ops.release_workspaces()
    assert not wrong and len(seen) == 20
    assert seen == sorted(set(seen))  # launched in the order of their tags
