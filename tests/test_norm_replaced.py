"""What a program has replaced is called: a norm, in the float32 mode, instead of norming inside the product behind it; a feed-forward's
activation."""
from types import SimpleNamespace

import pytest
import torch

import qwen_engine_amd  # noqa: F401
from qwen_engine_amd.parts.base import Stream, StreamInput
from qwen_engine_amd.parts import mlp
from qwen_engine_amd.parts.mlp import SwiGLU
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


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("how", ["class", "part", "derived"])
def test_a_replaced_activation_is_called(monkeypatch, dtype, how):
    """With the norm inside the product it would be passed by: it gets the rows that the norm's own kernel makes."""
    products = []
    fake = SimpleNamespace(gemm_norm_preferred=lambda rows, w, parts: True, gemm_branch_splits=lambda a, w: 0, EPI_SILU_MUL=2, EPI_SILU_MUL_IL=4,
                           gemm=lambda x, w, b=None, **kw: products.append(kw) or x)
    monkeypatch.setattr(mlp, "ops", fake)
    rows = torch.ones(2, 8)
    norm = SimpleNamespace(forward=lambda h, rt, delta=None: rows)
    ffn = SwiGLU(SimpleNamespace(intermediate_size=32, names=("gate", "up", "down")), 8)
    ffn.w_gu, ffn.w_down, ffn.interleaved = torch.zeros(64, 8, dtype=dtype), torch.zeros(8, 32, dtype=dtype), True
    x = StreamInput(Stream(torch.zeros(2, 8), torch.zeros(2, 8)), None, norm, torch.ones(8), 1e-6, SimpleNamespace(dtype=dtype))
    ffn.forward(x, None)
    assert products[0].get("norm_weight") is x.weight            # (as it is written: one product does it all)
    seen, mine = [], lambda x: seen.append(x) or x
    if how == "class":
        monkeypatch.setattr(SwiGLU, "activation", lambda self, x: mine(x))
    elif how == "part":
        ffn.activation = mine
    else:
        ffn.__class__ = type("Derived", (SwiGLU,), {"activation": lambda self, x: mine(x)})
    ffn.forward(x, None)
    assert seen == [rows]
