"""Which steps project their input in the step's kernel (pararnn_amd.decode): only
a plain, unwatched nn.Linear on rows that the kernel can read as they are; every
other form keeps the module's own call."""

import pytest
import torch
from torch import nn
from torch.utils.flop_counter import FlopCounterMode

from pararnn_amd import decode as D


def _ask(proj, x, out=None, d=16, gates=4, fused=True):
    return D._projects(proj, x, d, gates, fused, torch.zeros(x.shape[0], 64) if out is None else out)


def test_a_plain_linear_is_taken_in_every_storage_type():
    for dtype in (torch.float32, torch.bfloat16, torch.float16):
        lin = nn.Linear(16, 64).to(dtype)
        assert _ask(lin, torch.zeros(3, 16, dtype=dtype))
    assert _ask(nn.Linear(16, 64, bias=False), torch.zeros(3, 16))


class _Sub(nn.Linear):
    pass


class _Tensor(torch.Tensor):
    pass


def _hooked():
    lin = nn.Linear(16, 64)
    lin.register_forward_hook(lambda *a: None)
    return lin


def _patched():
    lin = nn.Linear(16, 64)
    lin.forward = lambda x: x
    return lin


def _parametrized():
    lin = nn.Linear(16, 64)
    nn.utils.parametrizations.weight_norm(lin)
    return lin


def _strided_weight():
    lin = nn.Linear(16, 64)
    lin.weight = nn.Parameter(torch.zeros(16, 64).t())
    return lin


@pytest.mark.parametrize("make", [lambda: None, lambda: nn.Identity(), lambda: _Sub(16, 64), _hooked,
                                  _patched, _parametrized, _strided_weight,
                                  lambda: nn.Linear(16, 60), lambda: nn.Linear(8, 64),
                                  lambda: nn.Linear(16, 64).bfloat16()])
def test_other_projections_keep_their_own_call(make):
    assert not _ask(make(), torch.zeros(3, 16))


@pytest.mark.parametrize("x", [torch.zeros(3, 32)[:, ::2], torch.zeros(16, 3).t(),
                               torch.zeros(49)[1:].view(3, 16), torch.zeros(0, 16),
                               torch.zeros(3, 16).as_subclass(_Tensor),
                               torch._neg_view(torch.zeros(3, 16))])
def test_other_inputs_keep_the_modules_call(x):
    assert not _ask(nn.Linear(16, 64), x)


def test_rows_of_a_partial_16_byte_word_and_overlapping_outputs():
    assert not _ask(nn.Linear(6, 64), torch.zeros(2, 6))
    assert not _ask(nn.Linear(20, 64).half(), torch.zeros(2, 20).half())
    buf = torch.zeros(4, 64)
    x = buf.view(-1)[:48].view(3, 16)
    assert not _ask(nn.Linear(16, 64), x, out=buf)
    assert not _ask(nn.Linear(16, 64), x, out=buf.view(-1)[40:].view(1, -1))
    assert _ask(nn.Linear(16, 64), x, out=buf.view(-1)[48:].view(1, -1))


def test_modes_autocast_and_global_hooks(monkeypatch):
    lin, x = nn.Linear(16, 64), torch.zeros(3, 16)
    with monkeypatch.context() as m:  # autocast of a device that is not here stays off
        m.setattr(torch, "is_autocast_enabled", lambda device_type=None: device_type == "cuda")
        assert not _ask(lin, x)
    with FlopCounterMode(display=False):
        assert not _ask(lin, x)
    with torch.device("cpu"):
        assert not _ask(lin, x)
    handle = nn.modules.module.register_module_forward_hook(lambda *a: None)
    try:
        assert not _ask(lin, x)
    finally:
        handle.remove()
    assert _ask(lin, x)


def test_large_steps_keep_the_library():
    assert D._small_step(64, 1024, 1024, 2, True) and not D._small_step(128, 1024, 1024, 2, True)
    assert D._small_step(16, 1024, 1024, 4, True) and not D._small_step(16, 1024, 1024, 4, False)
    assert D._small_step(512, 64, 64, 4, False) and not D._small_step(64, 1024, 1024, 4, True)


@pytest.mark.parametrize("d_in,rows,dtype", [(6, 2, torch.float32), (555, 3, torch.bfloat16),
                                             (1024, 4096, torch.float32)])
def test_sizes_are_told_before_anything_is_looked_at(d_in, rows, dtype, monkeypatch):
    """Rows of a partial 16-byte word and large steps keep the library call without the
    cost of the other checks."""
    def looked(*a, **k):
        raise AssertionError("looked further")

    monkeypatch.setattr(torch, "is_autocast_enabled", looked)
    monkeypatch.setattr(nn.modules.module, "_has_any_global_hook", looked)
    lin = nn.Linear(d_in, 64).to(dtype)
    assert not D._projects(lin, torch.zeros(rows, d_in, dtype=dtype), 16 if d_in < 1024 else 1024,
                           4, True, torch.zeros(1))
