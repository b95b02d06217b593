"""Attention over one cached latent per token.

Per token the cache holds c = norm(W_dkv x)[:R] (R = kv_rank) and one rotated key part of Dr numbers that
all heads share; a head's key is [Uk_h c | rotated part], its value Uv_h c.  The cache never holds expanded keys
or values, and single tokens need none: with q'_h = Uk_h^T q_h the score of head h against token j is
q'_h . c_j + q_rot_h . k_rot_j, one dot product against the cached row, and the head's output is
Uv_h (sum_j p_j c_j).  So the attention kernel sees one key/value head of R + Dr numbers whose first R are also
the value, read by all query heads, and the two maps are products per head before and after it (``ops.gemm_heads``).

Portions of prompts may do otherwise: rows that share their keys with some dozens of others cost less with the keys
and values expanded once for all of them (``ops.latent_prefill``).  Which rows go that way follows from the number of
(row, key) pairs a key has part in.

Queries come straight from the input (``q``), or through a normed latent of their own (``dq``, ``dq.norm``,
``uq``).  With ``output_gate`` the heads' outputs are multiplied by sigmoid(W_g x) before ``o``, a number per output
or (``gate_per_head``) per head.  A window, a learned sink per head (``sink``) and the pairing of the rotation
(neighbouring or half-split, by the kind of the position part) are parameters of the kernels.  A layer without a
latent of its own (``own_latent`` False) reads the cache of the schedule entry it is bound to.
"""
from __future__ import annotations

from typing import Dict, List, Optional, Tuple

import torch

from ..cache.plan import KVNeed
from ..kernels import ops
from .attention import prefill_tiles
from .base import CacheBinding, Runtime, TensorInfo
from .registry import build_part, register_part

# Bytes that the gathered cache rows and the expanded keys and values of a step may take, all its portions together (they are gone
# when the layer is done; a recorded step keeps them for its replays, and they count among what it holds)
EXPAND_MAX_BYTES = 1 << 30


class LatentAttention:
    graph_safe = True

    # ---- what the step function prepares for this part (parts.base) --------------------------
    # A step run as it comes knows its portions (ctx.seqs); a recorded portion is recorded for the number of keys that its
    # buffers hold, and where the keys lie the kernels read from the positions; single tokens beside a portion in a recorded
    # step go with the folded maps, all rows alike (its portion's first row and number of rows, which the lists of expanded keys
    # name, differ from replay to replay; unrecorded, a long portion beside single tokens is expanded).
    @staticmethod
    def step_extras(seqs) -> dict:
        return {"eager": 1}

    @staticmethod
    def portion_graph_key(tokens: int, keys: int) -> int:
        """The portion's keys rounded up to its rows times a power of two: few recorded steps for a prompt in many portions (each
        serves the places of more than half as many keys)."""
        n = int(tokens)
        while n < keys:
            n *= 2
        return n

    @staticmethod
    def portion_graph_extras(tokens: int, device, key: int) -> dict:
        return {"keys": int(key)}

    mixed_graph_dynamic_size = 0

    @staticmethod
    def mixed_graph_key(max_dec_position: int, portion_keys: int) -> int:
        return 0

    @staticmethod
    def mixed_graph_dynamic(rows: int, pad: int, tokens: int) -> List[int]:
        return []

    @staticmethod
    def mixed_graph_extras(rows: int, tokens: int, key, device, dynamic: torch.Tensor) -> dict:
        return {}

    def _seen(self, rows: int, keys: int) -> int:
        """How many of ``keys`` positions the last ``rows`` of them see."""
        return min(keys, self.window + rows - 1) if self.window else keys

    def _expanded_bytes(self, keys: int) -> int:
        return 2 * (-(-keys // 64) * 64) * (self.h * (self.dn + self.dv) + self.r + self.dr)

    def _pays(self, rows: int, keys: int, expanded: int = 0) -> bool:
        """True if rows that are the last of ``keys`` positions are better off with expanded keys: every key (``expanded`` of them,
        if those are more than the rows see) costs R (Dn + Dv) multiply-adds a head at some 500 TFLOP/s, which every pair of a
        row and a key pays back with the difference of 2 R + Dr at 200 and Dn + Dr + Dv at 350 (the rates of the kernels; half as
        much again asked for, the launches being more)."""
        seen = self._seen(rows, keys)
        pairs = rows * min(self.window, seen - rows / 2.0) if self.window else rows * (seen - rows / 2.0)
        a_key = self.r * (self.dn + self.dv) / 500.0
        a_pair = (2 * self.r + self.dr) / 200.0 - (self.dn + self.dr + self.dv) / 350.0
        return a_pair > 0 and pairs * a_pair > 1.5 * max(seen, expanded) * a_key

    def _expansion(self, ctx) -> Optional[dict]:
        """Which of the step's rows see expanded keys, made once per step for all layers of the same sizes: the rows' ranges, the
        others' ranges, and the lists that the kernels take."""
        if not ops.latent_prefill_supported(self.r, self.dn, self.dr, self.dv, ctx.rt.dtype):
            return None
        key = ("latent_attention.expansion", self.r, self.dn, self.dr, self.dv, self.h, self.window)
        if key not in ctx.memo:
            ex = next((ctx.extras[cls] for cls in type(self).__mro__ if cls in ctx.extras), {})
            wanted: List[Tuple[int, int, int]] = []                  # (first row, rows, keys)
            if "keys" in ex:                                         # a recorded portion: for all the places that replay it
                n, k = ctx.num_tokens, ex["keys"]
                if self._pays(n, k if k == n else k // 2 + 1, self._seen(n, k)):
                    wanted.append((0, n, self._seen(n, k)))
            elif "eager" in ex:
                for s in ctx.seqs:
                    if s.q_len > 1 and self._pays(s.q_len, s.kv_before + s.q_len):
                        wanted.append((s.q_start, s.q_len, self._seen(s.q_len, s.kv_before + s.q_len)))
            portions, room = [], EXPAND_MAX_BYTES
            for first, rows, keys in wanted:
                if self._expanded_bytes(keys) <= room:
                    room -= self._expanded_bytes(keys)
                    portions.append((first, rows, keys))
            ctx.memo[key] = self._lists(ctx, portions) if portions else None
        return ctx.memo[key]

    def _lists(self, ctx, portions: List[Tuple[int, int, int]]) -> dict:
        table, owner, tiles, group_portion, others = [], [], [], [], []
        done = 0
        for i, (first, rows, keys) in enumerate(portions):
            table += [first, rows, 64 * len(owner)]
            owner += [i] * (-(-keys // 64))
            mine = prefill_tiles([(first, rows)], 32)
            tiles += mine
            group_portion += [i] * (len(mine) // 8)
            if first > done:
                others.append((done, first))
            done = first + rows
        if done < ctx.num_tokens:
            others.append((done, ctx.num_tokens))
        flat = torch.tensor(table + owner + tiles + group_portion, dtype=torch.int32).to(ctx.rt.device)
        a, b, c = len(table), len(table) + len(owner), len(table) + len(owner) + len(tiles)
        return {"ranges": [(f, f + n) for f, n, _ in portions], "others": others, "portions": flat[:a].view(-1, 3),
                "owner": flat[a:b], "tiles": flat[b:c].view(-1, 2), "group_portion": flat[c:]}

    def __init__(self, spec, hidden_size: int):
        self.spec = spec
        self.hidden = int(hidden_size)
        self.h, self.dn, self.dr, self.dv = int(spec.num_heads), int(spec.head_dim), int(spec.rot_dim), int(spec.v_head_dim)
        self.r = int(spec.kv_rank)
        self.q_rank = int(spec.q_rank) if spec.q_rank else 0
        self.gated = bool(spec.output_gate)
        self.gate_per_head = bool(getattr(spec, "gate_per_head", False))
        self.window = int(spec.window) if getattr(spec, "window", None) else 0
        self.has_sink = bool(getattr(spec, "sink", False))
        self.own_latent = bool(getattr(spec, "own_latent", True))
        self.scale = float(spec.scale)
        self.eps = float(spec.norm_eps)
        self.position = build_part(spec.position, hidden_size) if spec.position is not None else None
        self.half_split = spec.position is not None and spec.position.kind == "rope_half_angles"
        self.sink = None
        self.w_q = self.w_dq = self.w_uq = self.q_norm = self.w_dkv = self.kv_norm = None
        self.w_uk_t = self.w_uv = self.w_g = self.w_o = None
        self._no_turn: Optional[torch.Tensor] = None
        self._w_uk: Optional[torch.Tensor] = None

    # ---- what it needs --------------------------------------------------------------------------
    @staticmethod
    def expected_tensors(spec, hidden: int) -> Dict[str, TensorInfo]:
        h, dq, dv, r = spec.num_heads, spec.head_dim + spec.rot_dim, spec.v_head_dim, spec.kv_rank
        t = {
            "uk": TensorInfo((h * spec.head_dim, r)),
            "uv": TensorInfo((h * dv, r)),
            "o": TensorInfo((hidden, h * dv)),
        }
        if getattr(spec, "own_latent", True):
            t["dkv"] = TensorInfo((r + spec.rot_dim, hidden))
            t["dkv.norm"] = TensorInfo((r,), "ones", "vector")
        if getattr(spec, "sink", False):
            t["sink"] = TensorInfo((h,), "zeros", "vector")
        if spec.q_rank:
            t["dq"] = TensorInfo((spec.q_rank, hidden))
            t["dq.norm"] = TensorInfo((spec.q_rank,), "ones", "vector")
            t["uq"] = TensorInfo((h * dq, spec.q_rank))
        else:
            t["q"] = TensorInfo((h * dq, hidden))
        if spec.output_gate:
            t["g"] = TensorInfo((h if getattr(spec, "gate_per_head", False) else h * dv, hidden))
        return t

    @staticmethod
    def cache_need(spec) -> Optional[KVNeed]:
        """One row of R + Dr numbers a token; with a window the cache keeps the window's keys, or ``keep_window``
        where later layers that read this cache look further back."""
        window = getattr(spec, "window", None)
        if window is not None and getattr(spec, "keep_window", None) is not None:
            window = max(int(window), int(spec.keep_window))
        return KVNeed(num_kv_heads=1, head_dim=spec.kv_rank + spec.rot_dim, window=window, planes=1)

    @staticmethod
    def state_need(spec, hidden: int):
        return None

    # ---- weights -----------------------------------------------------------------------------------
    def load(self, tensors: Dict[str, torch.Tensor], rt: Runtime) -> None:
        if self.q_rank:
            self.w_dq = rt.place_matrix(tensors["dq"])
            self.q_norm = rt.place_vector(tensors["dq.norm"])
            self.w_uq = rt.place_matrix(tensors["uq"])
        else:
            self.w_q = rt.place_matrix(tensors["q"])
        if self.own_latent:
            self.w_dkv = rt.place_matrix(tensors["dkv"])
            self.kv_norm = rt.place_vector(tensors["dkv.norm"])
        if self.has_sink:
            self.sink = rt.place_vector(tensors["sink"])
        # the key map per head, transposed: q' = Uk_h^T q is then a product against [R, dn] rows
        uk = tensors["uk"].view(self.h, self.dn, self.r)
        self.w_uk_t = rt.place_matrix(uk.transpose(1, 2).contiguous()) if self.dn > 0 else None
        # (and as it is, for expanded keys; a step uses one of the two)
        self._w_uk = rt.place_matrix(tensors["uk"]) if ops.latent_prefill_supported(self.r, self.dn, self.dr, self.dv, rt.dtype) else None
        self.w_uv = rt.place_matrix(tensors["uv"].view(self.h, self.dv, self.r))
        if self.gated:
            self.w_g = rt.place_matrix(tensors["g"])
        self.w_o = rt.place_matrix(tensors["o"])
        if self.position is not None:
            self.position.load({}, rt)
        self._no_turn = torch.zeros(0, dtype=torch.float32, device=rt.device)

    # ---- one step ------------------------------------------------------------------------------------
    def forward(self, x: torch.Tensor, ctx, binding: CacheBinding) -> torch.Tensor:
        """x [T, H] in the activation type.  Returns the mixer's output [T, H], or float32 partial
        products [S, T, H] of it."""
        if binding.kv is None:
            raise RuntimeError("latent attention was given no cache")
        T, dt = x.shape[0], ctx.rt.dtype
        g, cache = binding.group, binding.kv
        inv_freq = self.position.inv_freq() if self.position is not None else self._no_turn
        # queries
        if self.q_rank:
            cq = ops.rmsnorm(ops.gemm(x, self.w_dq, out_dtype=torch.float32), self.q_norm, self.eps, dt)
            q = ops.gemm(cq, self.w_uq)
        else:
            q = ops.gemm(x, self.w_q)
        q = q.view(T, self.h, self.dn + self.dr)
        if binding.write and not self.own_latent:
            raise RuntimeError("latent attention: a layer without a latent of its own has nothing to write into a cache")
        kv = ops.gemm(x, self.w_dkv, out_dtype=torch.float32) if binding.write else None
        o = torch.empty((T, self.h, self.dv), dtype=dt, device=x.device)
        gate = ops.gemm(x, self.w_g) if self.gated else None
        plan = self._expansion(ctx)
        if plan is None:
            self._folded(q, kv, ctx, binding, inv_freq, o, gate, 0, T)
        else:
            if kv is not None:
                ops.latent_kv_store(kv, self.kv_norm, self.eps, ctx.positions, inv_freq, ctx.slots[g], cache,
                                    half_split=self.half_split)
            for a, b in plan["others"]:
                self._folded(q[a:b], None, ctx, binding, inv_freq, o[a:b], None if gate is None else gate[a:b], a, b)
            for a, b in plan["ranges"]:
                ops.latent_q_rotate(q[a:b], ctx.positions[a:b], inv_freq, q[a:b], self.dn, half_split=self.half_split)
            ck, kr = ops.latent_gather(cache, ctx.positions, ctx.tok_seq, ctx.block_tables[g], plan["portions"], plan["owner"],
                                       self.r, window=self.window)
            kx = ops.gemm(ck, self._w_uk)
            vt = ops.gemm(self.w_uv.view(self.h * self.dv, self.r), ck)
            ops.latent_prefill(q, kx, kr, vt, o, plan["tiles"], plan["group_portion"], plan["portions"], ctx.positions, self.scale,
                               window=self.window, sink=self.sink, gate=gate)
        o = o.view(T, self.h * self.dv)
        splits = ops.gemm_branch_splits(o, self.w_o)
        if splits:
            return ops.gemm(o, self.w_o, epilogue=ops.EPI_PARTIAL, splits=splits)
        return ops.gemm(o, self.w_o)

    def _folded(self, q, kv, ctx, binding: CacheBinding, inv_freq, o, gate, a: int, b: int) -> None:
        """Rows a .. b of the step with the maps folded into the queries: o[t, h] = Uv_h sum_j p_j c_j.  kv: the rows' projections
        that are still to be normed, turned and written to the cache, or None."""
        g, cache = binding.group, binding.kv
        positions, tok_seq = ctx.positions[a:b], ctx.tok_seq[a:b]
        # the token's cache row (normed latent | rotated shared key part) and the rotated parts of the packed
        # queries [Uk^T q | rotated q], in one launch
        qp = torch.empty((b - a, self.h, self.r + self.dr), dtype=q.dtype, device=q.device)
        if kv is not None:
            ops.latent_kv_store(kv, self.kv_norm, self.eps, positions, inv_freq, ctx.slots[g][a:b], cache, q, qp, self.dn,
                                half_split=self.half_split)
        else:
            ops.latent_q_rotate(q, positions, inv_freq, qp, self.dn, half_split=self.half_split)
        if self.dn > 0:
            ops.gemm_heads(q, self.w_uk_t, qp)
        else:
            qp[:, :, :self.r].zero_()
        o_lat = ops.latent_attention(qp, cache, positions, tok_seq, ctx.block_tables[g], self.r, self.scale,
                                     window=self.window, sink=self.sink)
        ops.gemm_heads(o_lat, self.w_uv, o, gate)


register_part("latent_attention", LatentAttention)
