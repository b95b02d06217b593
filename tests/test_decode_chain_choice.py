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
