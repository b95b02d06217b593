"""Which rows of a step see expanded keys in latent attention: the plan alone, on the host."""
from types import SimpleNamespace

import pytest
import torch

import qwen_engine_amd  # noqa: F401
from qwen_engine_amd.config.spec import LatentAttentionSpec
from qwen_engine_amd.parts import latent_attention as L


@pytest.fixture()
def part(monkeypatch):
    monkeypatch.setattr(L.ops, "latent_prefill_supported", lambda *a: True)

    def make(window=None, heads=16):
        spec = LatentAttentionSpec(num_heads=heads, head_dim=128, rot_dim=64, v_head_dim=128, kv_rank=512, scale=0.1, norm_eps=1e-5,
                                   q_rank=None, window=window)
        return L.LatentAttention(spec, 256)

    return make


def plan(part, portions=(), recorded=None):
    """portions: (tokens cached, new tokens); recorded: (rows, the keys it is recorded for)."""
    seqs, at = [], 0
    for before, n in portions:
        seqs.append(SimpleNamespace(q_start=at, q_len=n, kv_before=before))
        at += n
    extras = {"eager": 1} if recorded is None else {"keys": recorded[1]}
    ctx = SimpleNamespace(rt=SimpleNamespace(dtype=torch.bfloat16, device="cpu"), memo={}, extras={type(part): extras}, seqs=seqs,
                          num_tokens=at if recorded is None else recorded[0])
    return part._expansion(ctx)


def test_a_steps_portions_share_the_bytes_there_are(part, monkeypatch):
    p = part()
    portions = [(3000, 512), (0, 1), (3000, 512), (100, 1), (3000, 512)]
    one = p._expanded_bytes(3512)
    assert one == 2 * 3520 * (16 * 256 + 576)
    for room, taken in ((3 * one, [0, 513, 1026]), (3 * one - 1, [0, 513]), (one, [0]), (one - 1, [])):
        monkeypatch.setattr(L, "EXPAND_MAX_BYTES", room)
        got = plan(p, portions)
        assert ([a for a, _ in got["ranges"]] if got else []) == taken
        if got:
            rows = sorted(got["ranges"] + got["others"])
            assert rows[0][0] == 0 and rows[-1][1] == 1538 and all(a[1] == b[0] for a, b in zip(rows, rows[1:]))
            assert 64 * got["owner"].shape[0] * (16 * 256 + 576) * 2 <= room
    # a portion that no longer fits leaves its place to a smaller one
    monkeypatch.setattr(L, "EXPAND_MAX_BYTES", one + p._expanded_bytes(600))
    assert [a for a, _ in plan(p, [(3000, 512), (3000, 512), (0, 600)])["ranges"]] == [0, 1024]


@pytest.mark.parametrize("window", [None, 300])
def test_few_rows_and_single_tokens_stay_folded(part, window):
    assert plan(part(window), [(4000, 1), (4000, 16), (0, 40)]) is None
    assert plan(part(window), [(0, 2048), (10, 1)])["others"] == [(2048, 2049)]
    seen = 64 * plan(part(window), [(4000, 512)])["owner"].shape[0]
    assert seen == (64 * -(-4512 // 64) if not window else 64 * -(-811 // 64))


@pytest.mark.parametrize("window", [None, 300, 5000])
@pytest.mark.parametrize("rows", [64, 96, 120, 128, 160, 256, 512, 2048])
def test_a_recorded_portion_pays_at_every_place_it_serves(part, rows, window):
    """Recorded for its rows times a power of two, it expands that many keys wherever it is replayed: with half as many keys seen it
    must still be worth it."""
    p = part(window)
    for doublings in range(7):
        keys = rows << doublings
        got = plan(p, recorded=(rows, keys))
        served = [n for n in range(rows, keys + 1) if p.portion_graph_key(rows, n) == keys]
        assert served[-1] == keys and len(served) == (1 if doublings == 0 else keys // 2)
        for n in (served[0], served[-1]):
            seen, expanded = p._seen(rows, n), p._seen(rows, keys)
            pairs = sum(min(i + 1, window or i + 1) for i in range(n - rows, n))
            gain = pairs * ((2 * 512 + 64) / 200 - 320 / 350)        # (microseconds' worth of folded minus expanded pairs, and of keys)
            assert got is None or gain > expanded * 512 * 256 / 500
            assert got is None or 64 * got["owner"].shape[0] >= seen
    assert plan(p, recorded=(512, 2048)) is not None
