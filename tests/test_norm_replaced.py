"""What a program has replaced is called: a norm, in the float32 mode, instead of norming inside the product behind it; a feed-forward's
activation, what an attention part does with q.  A part's forward, in the float32 mode,
gets the normed rows."""
from types import SimpleNamespace

import pytest
import torch

import qwen_engine_amd  # noqa: F401
from qwen_engine_amd.parts.base import Stream, StreamInput
from qwen_engine_amd.parts import attention, mlp
from qwen_engine_amd.parts.attention import PagedAttention
from qwen_engine_amd.parts.block import PreNormBlock
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


@pytest.mark.parametrize("how", ["class", "part", "derived"])
def test_a_replaced_attend_is_called(monkeypatch, how):
    """Steps of single tokens whose norm, rotation and cache write are inside the attention kernel have no q to hand on: they go one by one."""
    one, q = [], torch.ones(2, 4, 16)
    fake = SimpleNamespace(gemm=lambda x, w, b=None, **kw: x, gemm_qkv_supported=lambda *a: False, gemm_partial_preferred=lambda *a: False,
                           gemm_branch_splits=lambda *a: 0, attention_decode_fused_supported=lambda *a: True,
                           attention_decode_fused_preferred=lambda *a: True, qk_rope_store=lambda *a: q,
                           attention_decode_fused=lambda *a, **kw: one.append(a) or q)
    monkeypatch.setattr(attention, "ops", fake)
    part = PagedAttention(SimpleNamespace(num_heads=4, num_kv_heads=2, head_dim=16, scale=0.25, window=None, qk_norm_eps=None, position=None), 64)
    ctx = SimpleNamespace(positions=None, tok_seq=None, block_tables=[None], slots=[None], shared_keys=None, max_position=9, page_size=16, memo={},
                          extras={PagedAttention: {"dec_tokens": torch.zeros(2, dtype=torch.int32), "other_tokens": None, "max_dec_position": 9}})
    binding = SimpleNamespace(kv=torch.zeros(1, 2, 2, 16, 16), group=0, write=True)
    part.forward(torch.zeros(2, 64), ctx, binding)
    assert len(one) == 1
    seen, mine = [], lambda q, ctx, cache, g, T: seen.append(q) or q
    if how == "class":
        monkeypatch.setattr(PagedAttention, "_attend", lambda self, *a: mine(*a))
    elif how == "part":
        part._attend = mine
    else:
        part.__class__ = type("Derived", (PagedAttention,), {"_attend": lambda self, *a: mine(*a)})
    part.forward(torch.zeros(2, 64), ctx, binding)
    assert len(one) == 1 and len(seen) == 1 and seen[0] is q


@pytest.mark.parametrize("part", [SwiGLU, PagedAttention])
@pytest.mark.parametrize("how", ["class", "part", "derived"])
@pytest.mark.parametrize("delta", [None, torch.zeros(2, 8), torch.zeros(1, 2, 8)])
def test_a_replaced_forward_gets_the_normed_rows(monkeypatch, part, how, delta):
    rows, norm = torch.ones(2, 8), RMSNorm(SimpleNamespace(eps=1e-6), 8)
    norm.forward = lambda h, rt, delta=None: rows
    ctx, one = SimpleNamespace(rt=SimpleNamespace(dtype=torch.float32)), object.__new__(part)
    given = lambda: PreNormBlock._input(norm, one, Stream(torch.zeros(2, 8), torch.zeros(2, 8)), delta, ctx)
    assert isinstance(given(), StreamInput)
    if how == "class":
        monkeypatch.setattr(part, "forward", lambda self, *a: None)
    elif how == "part":
        one.forward = lambda *a: None
    else:
        one = object.__new__(type("Derived", (part,), {"forward": lambda self, *a: None}))
    assert given() is rows
    ctx.rt.dtype = torch.bfloat16                  # (there a part that says it takes the stream gets it, as it always did)
    assert isinstance(given(), StreamInput) == (delta is None or delta.dim() == 3)


def test_recorded_steps_of_a_derived_class(monkeypatch):
    """What a class prepares for its recorded mixed steps need not hold every row: single tokens beside a portion in one launch make the list then."""
    fake = SimpleNamespace(attention_prefill_supported=lambda *a: True, prefill_uncut_keys=lambda: 1024, prefill_takes_single=lambda *a: True,
                           prefill_tile_rows=lambda *a: 16, prefill_tiles_on_device=lambda *a: "tiles")
    monkeypatch.setattr(attention, "ops", fake)
    part, i32 = object.__new__(PagedAttention), lambda n: torch.arange(n, dtype=torch.int32)
    part.hq = part.hkv = 4
    ex = {"dec_tokens": i32(3), "other_tokens": i32(8) + 3, "max_dec_position": 511, "other_keys_row": None, "portions": torch.zeros(2, 2), "portion_rows": 8}
    rows, tiles = part._all_tiles(SimpleNamespace(memo={}, num_tokens=11, seqs=[]), ex, torch.zeros(11, 4, 16), None)
    assert tiles == "tiles" and torch.equal(rows, i32(11))
    ex["all_tokens"] = i32(11)
    assert part._all_tiles(SimpleNamespace(memo={}, num_tokens=11, seqs=[]), ex, torch.zeros(11, 4, 16), None)[0] is ex["all_tokens"]
