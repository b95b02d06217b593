"""When the layers of a step go to one launch (``parts.chain``) and when they run one by one: on the CPU, with the launch itself replaced
by a note of what it was given."""
from types import SimpleNamespace

import pytest
import torch

import qwen_engine_amd  # noqa: F401
from qwen_engine_amd.config import config_from_dict
from qwen_engine_amd.kernels import ops
from qwen_engine_amd.parts import DecoderModel, Runtime, expected_tensors
from qwen_engine_amd.parts.attention import PagedAttention
from qwen_engine_amd.parts.base import CacheBinding
from qwen_engine_amd.parts.block import PreNormBlock
from qwen_engine_amd.parts.chain import run_as_chain
from qwen_engine_amd.parts.mlp import SwiGLU
from qwen_engine_amd.parts.norm import RMSNorm
from qwen_engine_amd.parts.rope import RotaryHalf
from tiny import TINY_F

CPU = torch.device("cpu")


@pytest.fixture
def step(monkeypatch):
    """A model with the sizes of F, a step of two single tokens, and what the launch was given."""
    spec = config_from_dict(TINY_F).to_model_spec()
    model = DecoderModel(spec)
    model.load({n: torch.zeros(tuple(i.shape), dtype=torch.bfloat16) for n, i in expected_tensors(spec).items() if not i.optional},
               Runtime(CPU, torch.bfloat16))
    given = []
    monkeypatch.setattr(ops, "decode_chain_preferred", lambda *a: True)
    monkeypatch.setattr(ops, "decode_chain", lambda h, layers, *a, **kw: given.append((h, layers, a, kw)))
    i32 = lambda *x: torch.tensor(x, dtype=torch.int32)
    ctx = SimpleNamespace(rt=Runtime(CPU, torch.bfloat16), positions=i32(5, 40), tok_seq=i32(0, 1), block_tables=[i32(0, 0, 0).view(1, 3)] * 2,
                          slots=[i32(5, 40)] * 2, shared_keys=None, late=None, max_position=40, memo={},
                          extras={PagedAttention: {"dec_tokens": i32(0, 1), "other_tokens": i32(), "max_dec_position": 40}})
    bindings = [[CacheBinding(kv=torch.zeros(3, 2, 2, 16, 128, dtype=torch.bfloat16), group=0, write=True, state=None)] for _ in spec.schedule]
    return SimpleNamespace(blocks=model.blocks, schedule=spec.schedule, h=torch.zeros(2, 256), ctx=ctx, bindings=bindings, given=given,
                           run=lambda s: run_as_chain(s.blocks, s.schedule, s.h, s.ctx, s.bindings))


def test_a_later_layer_that_keeps_nothing(step):
    """A block of another kind may have no cache at all, and so no binding."""
    class Other:
        pass
    step.blocks[2], step.bindings[2] = Other(), []
    assert not step.run(step) and not step.given


@pytest.mark.parametrize("cls,name", [(PagedAttention, "forward"), (PagedAttention, "_project_out"), (SwiGLU, "forward"), (SwiGLU, "activation"),
                                      (RMSNorm, "forward"), (PreNormBlock, "forward"), (RotaryHalf, "table")])
@pytest.mark.parametrize("whole_class", [True, False])
def test_methods_that_a_program_has_replaced(step, monkeypatch, cls, name, whole_class):
    """A trace put around a method, of all parts of a class or of one, is called: the layers run one by one."""
    assert step.run(step) and len(step.given) == 1
    real = getattr(cls, name)
    if whole_class:
        monkeypatch.setattr(cls, name, lambda *a, **kw: real(*a, **kw))
    else:
        b = step.blocks[1]
        part = {PagedAttention: b.mixer, SwiGLU: b.ffn, RMSNorm: b.ffn_norm, PreNormBlock: b, RotaryHalf: b.mixer.position}[cls]
        setattr(part, name, lambda *a, **kw: real(part, *a, **kw))
    assert not step.run(step) and len(step.given) == 1


def test_what_the_launch_is_given(step):
    assert step.run(step)
    (h, layers, args, more), = step.given
    c, b, mixers = step.ctx, step.blocks, [x.mixer for x in step.blocks]
    assert h is step.h and len(layers) == 3
    for L, x, (binding,) in zip(layers, b, step.bindings):
        assert L["w_qkv"] is x.mixer.w_qkv and L["w_o"] is x.mixer.w_o and L["w_gu"] is x.ffn.w_gu and L["w_down"] is x.ffn.w_down
        assert L["norm1"] is x.mixer_norm.weight and L["norm2"] is x.ffn_norm.weight and L["q_norm"] is x.mixer.q_norm and L["k_norm"] is x.mixer.k_norm
        assert L["cache"] is binding.kv and (L["eps1"], L["eps2"]) == (x.mixer_norm.eps, x.ffn_norm.eps)
    assert args[:4] == (c.positions, c.tok_seq, c.block_tables[0], c.slots[0])
    assert args[4:8] == (4, mixers[0].scale, 40, mixers[0].qk_eps) and args[8] is mixers[0].position.table() and args[9] is None and more == {"late": None}


def _float32_step(s):
    s.ctx.rt = Runtime(CPU, torch.float32)


def _some_rows_are_a_prompts(s):
    s.ctx.extras[PagedAttention].update(dec_tokens=torch.tensor([0], dtype=torch.int32), other_tokens=torch.tensor([1], dtype=torch.int32))


def _derived_block(s):
    s.blocks[1].__class__ = type("Derived", (PreNormBlock,), {})


def _derived_mixer(s):
    s.blocks[1].mixer.__class__ = type("Derived", (PagedAttention,), {})


def _derived_feed_forward(s):
    s.blocks[1].ffn.__class__ = type("Derived", (SwiGLU,), {})


def _derived_norm(s):
    s.blocks[1].ffn_norm.__class__ = type("Derived", (RMSNorm,), {})


def _no_feed_forward(s):
    s.blocks[1].ffn = s.blocks[1].ffn_norm = None


def _window(s):
    s.blocks[1].mixer.window = 64


def _bias(name):
    def set_bias(s):
        part = s.blocks[1].ffn if name == "b_gu" else s.blocks[1].mixer
        setattr(part, name, torch.zeros(8))
    set_bias.__name__ = "_" + name
    return set_bias


def _gate_and_up_apart(s):
    s.blocks[1].ffn.interleaved = False


def _cache_of_another_group(s):
    s.bindings[1][0].group = 1


def _cache_of_another_layer(s):
    s.bindings[1][0].kv, s.bindings[1][0].write = s.bindings[0][0].kv, False


def _no_cache(s):
    s.bindings[1][0].kv = None


def _another_base(s):
    s.blocks[1].mixer.position.theta = 5e5


def _no_rotation_in_one(s):
    s.blocks[1].mixer.position = None


def _derived_rotation(s):
    for b in s.blocks:
        b.mixer.position.__class__ = type("Derived", (RotaryHalf,), {})


def _rotation_of_half_a_head(s):
    for b in s.blocks:
        b.mixer.position.rotary_dim, b.mixer.position._table = 64, b.mixer.position._table[:, :64].contiguous()


def _position_beyond_the_table(s):
    s.ctx.max_position = TINY_F["max_position_embeddings"]


def _another_scale(s):
    s.blocks[1].mixer.scale *= 2


def _another_eps(s):
    s.blocks[1].mixer.qk_eps = 1e-5


def _matrix_in_float32(s):
    s.blocks[1].ffn.w_down = s.blocks[1].ffn.w_down.float()


def _matrix_at_an_odd_address(s):
    w = s.blocks[1].mixer.w_o
    s.blocks[1].mixer.w_o = torch.zeros(w.numel() + 1, dtype=w.dtype)[1:].view(w.shape)


def _norm_at_an_odd_address(s):
    s.blocks[1].mixer.k_norm = torch.zeros(129)[1:]


@pytest.mark.parametrize("change", [
    _float32_step, _some_rows_are_a_prompts, _derived_block, _derived_mixer, _derived_feed_forward, _derived_norm, _no_feed_forward, _window,
    _bias("b_qkv"), _bias("b_o"), _bias("b_gu"), _gate_and_up_apart, _cache_of_another_group, _cache_of_another_layer, _no_cache, _another_base,
    _no_rotation_in_one, _derived_rotation, _rotation_of_half_a_head, _position_beyond_the_table, _another_scale, _another_eps, _matrix_in_float32,
    _matrix_at_an_odd_address, _norm_at_an_odd_address], ids=lambda f: f.__name__[1:])
def test_what_runs_one_by_one(step, change):
    """One layer that differs, or a step of another kind, is enough; nothing has been touched by then."""
    change(step)
    assert step.run(step) is False and not step.given
    assert not step.h.any() and not any(b[0].kv is not None and b[0].kv.any() for b in step.bindings)


def test_sizes_where_it_is_not_the_quicker_way(step, monkeypatch):
    asked = []
    monkeypatch.setattr(ops, "decode_chain_preferred", lambda *a: asked.append(a))
    assert not step.run(step) and not step.given and asked == [(2, 256, 4, 2, 128, 384, 16, 40)]
