"""The float32 mode calls a norm that a program has replaced instead of norming inside the product behind it."""
from types import SimpleNamespace

import pytest
import torch

import qwen_engine_amd  # noqa: F401
from qwen_engine_amd.parts.base import Stream, StreamInput
from qwen_engine_amd.parts.norm import RMSNorm

OPS = SimpleNamespace(gemm_norm_preferred=lambda rows, w, parts: True)


@pytest.mark.parametrize("delta", [None, torch.zeros(2, 8), torch.zeros(1, 2, 8)])
def test_a_replaced_norm_is_called(monkeypatch, delta):
    norm = RMSNorm(SimpleNamespace(eps=1e-6), 8)
    x = StreamInput(Stream(torch.zeros(2, 8), torch.zeros(2, 8)), delta, norm, torch.ones(8), 1e-6, SimpleNamespace(dtype=torch.float32))
    w = torch.zeros(4, 8)
    assert x.fusable() and x.prefers_prologue(OPS, w) and not x.prefers_prologue(OPS, w.bfloat16())
    written = RMSNorm.forward
    monkeypatch.setattr(RMSNorm, "forward", lambda self, *a, **k: written(self, *a, **k))
    assert not x.prefers_prologue(OPS, w)
    monkeypatch.undo()
    assert x.prefers_prologue(OPS, w)
    norm.forward = lambda *a, **k: None
    assert not x.prefers_prologue(OPS, w)
