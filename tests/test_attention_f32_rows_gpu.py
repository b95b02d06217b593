"""Float32 attention of many tokens, several to a block: a token's bits are those it has alone."""
import pytest
import torch

import qwen_engine_amd  # noqa: F401

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.fixture(scope="module")
def ops():
    from qwen_engine_amd.kernels import ops as o
    return o


@pytest.mark.parametrize("hq,hkv,D,P,softcap", [(8, 4, 128, 16, 0.0), (8, 1, 64, 16, 0.0), (6, 2, 128, 48, 0.0), (4, 4, 80, 16, 20.0), (10, 2, 32, 5, 0.0),
                                                (4, 2, 256, 16, 0.0)])
@pytest.mark.parametrize("portions", [[(300, 0)], [(1, 0), (70, 0), (3, 130), (1, 40), (121, 17), (2, 0), (140, 250)]])
@pytest.mark.parametrize("odd", [None, float("inf"), float("nan")])
def test_tokens_of_a_block_and_alone(ops, hq, hkv, D, P, softcap, portions, odd):
    """Portions (rows, keys before them) of several requests, whose edges lie inside blocks; what was never written is NaN.  A value that is infinite or
    NaN reaches the tokens that see it and no others."""
    g = torch.Generator().manual_seed(3)
    lens = [r + b for r, b in portions]
    pages = [-(-n // P) for n in lens]
    order = torch.randperm(sum(pages), generator=g).int()
    table, at = torch.full((len(lens), max(pages)), -1, dtype=torch.int32), 0
    cache = torch.full((sum(pages), 2, hkv, P * D), float("nan"))
    ks, vs = [], []
    for i, n in enumerate(lens):
        k, v = torch.randn(n, hkv, D, generator=g), torch.randn(n, hkv, D, generator=g)
        if odd is not None and i == len(lens) - 1:
            v[n - 20, 0, 5] = odd
        for j in range(pages[i]):
            part = slice(j * P, min(n, (j + 1) * P))
            page = cache[order[at + j]]
            page[0].view(hkv, P, D)[:, :part.stop - part.start] = k[part].transpose(0, 1)
            page[1].view(hkv, D, P)[:, :, :part.stop - part.start] = v[part].permute(1, 2, 0)
        table[i, :pages[i]] = order[at:at + pages[i]]
        at += pages[i]
        ks.append(k)
        vs.append(v)
    cache, table = cache.view(-1, 2, hkv, P, D).to(DEV), table.to(DEV)
    pos = [b + i for r, b in portions for i in range(r)]
    seq = [k for k, (r, _) in enumerate(portions) for _ in range(r)]
    T = len(pos)
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device=DEV)
    q = torch.randn(T, hq, D, generator=g)
    run = lambda which: ops.attention(q.to(DEV), cache, i32(pos), i32(seq), table, D ** -0.5, dec_tokens=i32([]), other_tokens=i32(which),
                                      softcap=softcap).cpu()
    every = run(range(T))
    for requests in (1, len(portions), T):       # (a hint: other forms, the same bits; NaN compares as NaN)
        hinted = ops.attention(q.to(DEV), cache, i32(pos), i32(seq), table, D ** -0.5, dec_tokens=i32([]), other_tokens=i32(range(T)), softcap=softcap,
                               other_requests=requests).cpu()
        assert torch.equal(hinted.nan_to_num(), every.nan_to_num()) and torch.equal(hinted.isnan(), every.isnan()), requests
    for t in sorted({0, 1, T // 2, T - 21, T - 20, T - 8, T - 1, *range(60, 80)}):
        alone = run([t])[t]
        assert torch.equal(torch.nan_to_num(every[t]), torch.nan_to_num(alone)) and torch.equal(every[t].isnan(), alone.isnan()), t
        if odd is None or seq[t] != len(lens) - 1 or pos[t] < lens[-1] - 20:
            k, v = ks[seq[t]][:pos[t] + 1].double(), vs[seq[t]][:pos[t] + 1].double()
            s = torch.stack([k[:, h * hkv // hq] @ q[t, h].double() for h in range(hq)]) * D ** -0.5
            w = torch.softmax(softcap * torch.tanh(s / softcap) if softcap else s, -1)
            want = torch.stack([w[h] @ v[:, h * hkv // hq] for h in range(hq)])
            assert float((every[t].double() - want).norm() / want.norm()) < 1e-5, t
        else:
            assert not every[t, 0, 5].isfinite()


@pytest.mark.parametrize("hq,hkv", [(8, 4), (8, 8), (20, 4)])
@pytest.mark.parametrize("counts", [[1] * 67, [2, 3] * 14, [4] * 40, [1, 9, 1, 5, 30, 1, 1, 2] * 4])
def test_many_requests_of_few_tokens(ops, hq, hkv, counts):
    """Blocks whose tokens belong to two to sixteen requests, some of which other blocks take: a token's bits are those it has alone."""
    D, P = 64, 16
    g = torch.Generator().manual_seed(len(counts))
    before = [(37 * i) % 90 for i in range(len(counts))]
    pages = [-(-(b + c) // P) for b, c in zip(before, counts)]
    table, at = torch.full((len(counts), max(pages)), -1, dtype=torch.int32), 0
    for i, n in enumerate(pages):
        table[i, :n] = torch.arange(at, at + n, dtype=torch.int32)
        at += n
    cache = torch.randn(at, 2, hkv, P, D, generator=g).to(DEV)
    pos = [b + j for b, c in zip(before, counts) for j in range(c)]
    seq = [i for i, c in enumerate(counts) for _ in range(c)]
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device=DEV)
    q, T = torch.randn(len(pos), hq, D, generator=g).to(DEV), len(pos)
    assert T * hkv > 256                     # (fewer have a block each)
    run = lambda which, **kw: ops.attention(q, cache, i32(pos), i32(seq), table.to(DEV), 0.1, dec_tokens=i32([]), other_tokens=i32(which), **kw)
    alone = torch.stack([run([t])[t] for t in range(T)])
    for requests in (0, 1, len(counts)):
        assert torch.equal(run(range(T), other_requests=requests), alone), requests
    assert torch.equal(ops.attention(q, cache, i32(pos), i32(seq), table.to(DEV), 0.1), alone)
    if max(counts) == 1:
        got = ops.attention(q, cache, i32(pos), i32(seq), table.to(DEV), 0.1, dec_tokens=i32(range(T)), max_dec_position=max(pos))
        assert torch.equal(got, alone)


def test_many_single_tokens_take_no_turns(ops):
    """Twice the tokens, each of a request of its own, take less than three times as long (with a block's requests one after another, six times)."""
    hq, hkv, D, P, keys = 16, 8, 128, 16, 400
    cache = torch.randn(64 * keys // P, 2, hkv, P, D, device=DEV)
    table = torch.arange(64 * keys // P, dtype=torch.int32, device=DEV).view(64, -1)
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device=DEV)
    q = torch.randn(64, hq, D, device=DEV)

    def took(n):
        rows, pos = i32(range(n)), i32([keys - 1] * 64)
        run = lambda: ops.attention(q, cache, pos, i32(range(64)), table, 0.1, dec_tokens=rows, max_dec_position=keys - 1)
        run()
        times = []
        for _ in range(5):
            a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            torch.cuda.synchronize()
            a.record()
            for _ in range(20):
                run()
            b.record()
            b.synchronize()
            times.append(a.elapsed_time(b))
        return min(times)
    assert took(64) < 3 * took(32)
