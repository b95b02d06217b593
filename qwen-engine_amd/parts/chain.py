"""The layers of a step of single new tokens in one launch (``ops.decode_chain``), where every layer of the schedule is
a plain pre-norm block: norm, attention over its own cache, norm, gated feed-forward, without biases or a window."""
from __future__ import annotations

from types import FunctionType
from typing import List

import torch

from ..kernels import ops
from .attention import PagedAttention
from .base import CacheBinding
from .block import PreNormBlock
from .mlp import SwiGLU
from .norm import RMSNorm
from .rope import RotaryHalf


def _methods(cls) -> dict:
    return {name: v for name, v in vars(cls).items() if isinstance(v, (FunctionType, staticmethod, classmethod, property))}


# What the chain knows the layers to do is what these classes do as they are written.  Where a program has put something else in the place of
# one of their methods (a trace, a change of its own), the layers run one by one and call it.
_WRITTEN = {cls: _methods(cls) for cls in (PreNormBlock, PagedAttention, SwiGLU, RMSNorm, RotaryHalf)}


def _as_written() -> bool:
    return all(_methods(cls) == methods for cls, methods in _WRITTEN.items())


def _is(part, cls) -> bool:
    """A part of this very class, with the class's methods."""
    return type(part) is cls and _WRITTEN[cls].keys().isdisjoint(vars(part))


def _of_all_layers(mixer, ffn):
    """What every layer has alike, or None: a position encoding that the chain does not know."""
    pos = mixer.position
    if pos is not None and not _is(pos, RotaryHalf):
        return None
    turn = None if pos is None else (pos.theta, pos.rotary_dim, pos.max_positions)
    return mixer.hq, mixer.hkv, mixer.d, mixer.scale, mixer.qk_eps, ffn.inter, turn


def run_as_chain(blocks, schedule, h: torch.Tensor, ctx, bindings: List[CacheBinding]) -> bool:
    """Runs the schedule's layers on the 32-bit stream h [T, H] in place and returns True, or returns False and
    leaves everything as it is: the layers are then run one by one."""
    T = h.shape[0]
    if ctx.rt.dtype != torch.bfloat16 or not schedule:
        return False
    one = blocks[schedule[0].layer]
    if not (_is(one, PreNormBlock) and _is(one.mixer, PagedAttention) and _is(one.ffn, SwiGLU)):
        return False
    mix, g = one.mixer, bindings[0][0].group
    ex = mix._extras(ctx)
    if ex["dec_tokens"] is None or ex["dec_tokens"].shape[0] != T or (ex["other_tokens"] is not None and ex["other_tokens"].shape[0]):
        return False
    kv = bindings[0][0].kv
    if kv is None or g is None or not ops.decode_chain_preferred(T, h.shape[1], mix.hq, mix.hkv, mix.d, one.ffn.inter, kv.shape[3],
                                                                 ex["max_dec_position"]):
        return False
    same = _of_all_layers(mix, one.ffn)
    table = mix.position.table() if mix.position is not None and same else None
    if same is None or (table is not None and (table.shape[1] != mix.d or ctx.max_position >= table.shape[0])):
        return False                       # (a position beyond the table: the layers say so)
    if not _as_written():
        return False
    layers = []
    for entry, users in zip(schedule, bindings):
        b = blocks[entry.layer]
        if not (_is(b, PreNormBlock) and _is(b.mixer, PagedAttention) and _is(b.ffn, SwiGLU) and
                _is(b.mixer_norm, RMSNorm) and _is(b.ffn_norm, RMSNorm)):
            return False
        m, f, c = b.mixer, b.ffn, users[0]
        if (c.kv is None or not c.write or c.group != g or m.window or m.b_qkv is not None or m.b_o is not None or f.b_gu is not None or
                not f.interleaved):
            return False
        if _of_all_layers(m, f) != same or not all(w.dtype == torch.bfloat16 and w.data_ptr() % 16 == 0
                                                   for w in (m.w_qkv, m.w_o, f.w_gu, f.w_down, c.kv)):
            return False
        if any(v is not None and v.data_ptr() % 16 for v in (b.mixer_norm.weight, b.ffn_norm.weight, m.q_norm, m.k_norm)):
            return False
        layers.append({"w_qkv": m.w_qkv, "w_o": m.w_o, "w_gu": f.w_gu, "w_down": f.w_down, "norm1": b.mixer_norm.weight,
                       "norm2": b.ffn_norm.weight, "q_norm": m.q_norm, "k_norm": m.k_norm, "cache": c.kv,
                       "eps1": b.mixer_norm.eps, "eps2": b.ffn_norm.eps})
    ops.decode_chain(h, layers, ctx.positions, ctx.tok_seq, ctx.block_tables[g], ctx.slots[g], mix.hq, mix.scale, ex["max_dec_position"],
                     mix.qk_eps if mix.qk_eps is not None else 0.0, table, ctx.shared_keys, late=ctx.late)
    return True
