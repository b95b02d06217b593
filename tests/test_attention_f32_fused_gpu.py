"""Float32 attention of single new tokens with norm, rotation and cache write inside: the bits, and the cache, of the kernels one by one.  What is
written nowhere counts for its own token all the same, which needs no page for it."""
import pytest
import torch

import qwen_engine_amd  # noqa: F401

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.fixture(scope="module")
def ops():
    from qwen_engine_amd.kernels import ops as o
    return o


# own keys first and last in a tile, alone in theirs, in a walk's first tile and in later ones; a page of the next tile untouched
POS = [0, 1, 15, 16, 17, 47, 112, 127, 128, 143, 500, 1100]


@pytest.mark.parametrize("hq,hkv,D,P,window", [(16, 8, 128, 16, 0), (8, 4, 64, 48, 0), (32, 2, 128, 16, 0), (6, 6, 80, 32, 0), (4, 2, 16, 16, 40)])
@pytest.mark.parametrize("steps", ["all", "no norm", "no rotation", "not written", "some not written", "some rows"])
def test_one_launch_and_two(ops, hq, hkv, D, P, window, steps):
    g = torch.Generator().manual_seed(hq * D + P)
    n = len(POS)
    pages = [p // P + 1 for p in POS]
    order, at = torch.randperm(sum(pages), generator=g).int(), 0
    table = torch.full((n, max(pages)), -1, dtype=torch.int32)
    cache = torch.full((sum(pages), 2, hkv, P * D), float("nan"))          # (a key tile [P][D], a value tile [D][P]; NaN where nothing was written)
    slots = []
    for i, p in enumerate(POS):
        ids = order[at:at + pages[i]]
        at += pages[i]
        table[i, :pages[i]] = ids
        slots.append(int(ids[p // P]) * P + p % P)
        for j in range(pages[i]):
            m = max(0, min(p - j * P, P))
            cache[ids[j], 0].view(hkv, P, D)[:, :m] = torch.randn(hkv, m, D, generator=g)
            cache[ids[j], 1].view(hkv, D, P)[:, :, :m] = torch.randn(hkv, D, m, generator=g)
    cache = cache.view(-1, 2, hkv, P, D).to(DEV)
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device=DEV)
    qkv = torch.randn(n, (hq + 2 * hkv) * D, generator=g).to(DEV)
    qw, kw = ((1 + 0.1 * torch.randn(D, generator=g)).to(DEV) for _ in range(2))
    rot = torch.randn(max(POS) + 1, D, generator=g).to(DEV)
    if steps == "no norm":
        qw = kw = None
    if steps == "no rotation":
        rot = None
    slots = i32(slots)
    pos, seq, table = i32(POS), i32(range(n)), table.to(DEV)
    assert ops.attention_decode_fused_supported(qkv, cache, hq, rot)
    two = cache.clone()
    q = ops.qk_rope_store(qkv, hq, hkv, D, pos, qw, kw, 1e-6, rot, slots, two, P)
    rows = i32(range(n))
    if steps == "some rows":                                 # (the cache is then written for those alone)
        rows = i32([3, 0, 11])
    want = ops.attention(q, two, pos, seq, table, D ** -0.5, window, dec_tokens=rows, max_dec_position=max(POS))
    one = cache.clone()
    if "not written" in steps:
        left = torch.arange(n, device=DEV) % 2 == 1 if steps == "some not written" else torch.ones(n, dtype=torch.bool, device=DEV)
        two = cache.clone()
        ops.qk_rope_store(qkv, hq, hkv, D, pos, qw, kw, 1e-6, rot, torch.where(left, -1, slots), two, P)
        for i, p in enumerate(POS):                          # (where a page would begin with the token, there is none)
            if left[i] and p % P == 0:
                table[i, p // P] = -1
        slots = None if bool(left.all()) else torch.where(left, -1, slots)
    got = ops.attention_decode_fused(qkv, hq, one, pos, seq, table, D ** -0.5, window, rows if steps == "some rows" else None, max(POS), qw, kw, 1e-6,
                                     rot, slots)
    assert bool(torch.isfinite(want[rows.long()]).all())
    assert torch.equal(got[rows.long()], want[rows.long()])
    if steps != "some rows":
        assert torch.equal(one.nan_to_num(7.0), two.nan_to_num(7.0))
    again = ops.attention_decode_fused(qkv, hq, one, pos, seq, table, D ** -0.5, window, rows, max(POS), qw, kw, 1e-6, rot, slots)
    assert torch.equal(again[rows.long()], want[rows.long()])


def test_what_is_not_taken(ops):
    qkv = lambda n, hq, hkv, D: torch.zeros(n, (hq + 2 * hkv) * D, device=DEV)
    cache = lambda hkv, P, D: torch.zeros(1, 2, hkv, P, D, device=DEV)
    assert not ops.attention_decode_fused_supported(qkv(33, 8, 8, 16), cache(8, 16, 16), 8, None)
    assert not ops.attention_decode_fused_supported(qkv(1, 34, 2, 16), cache(2, 16, 16), 34, None)
    assert not ops.attention_decode_fused_supported(qkv(1, 4, 2, 144), cache(2, 16, 144), 4, None)
    assert not ops.attention_decode_fused_supported(qkv(1, 4, 2, 16), cache(2, 5, 16), 4, None)
    assert not ops.attention_decode_fused_supported(qkv(1, 4, 2, 16), cache(2, 16, 16)[:0], 4, None)
    assert not ops.attention_decode_fused_supported(qkv(1, 4, 2, 16), cache(2, 16, 16).bfloat16(), 4, None)
