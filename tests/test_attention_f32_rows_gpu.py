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
