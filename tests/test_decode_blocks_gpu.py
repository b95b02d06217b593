"""Single new tokens whose keys one block walks (four waves, each with every fourth tile and a softmax of its own), in one segment and in several."""
import pytest
import torch

import qwen_engine_amd  # noqa: F401

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.fixture(scope="module")
def ops():
    from qwen_engine_amd.kernels import ops as o
    return o


def rand(*shape, seed=0):
    return torch.randn(*shape, generator=torch.Generator().manual_seed(seed))


def _requests(pos, hkv, D, P):
    """(cache, block table, keys and values of every request): shuffled pages, NaN wherever nothing was written."""
    pages = [p // P + 1 for p in pos]
    order = torch.randperm(sum(pages), generator=torch.Generator().manual_seed(7)).int()
    table, at = torch.full((len(pos), max(pages)), -1, dtype=torch.int32), 0
    cache = torch.full((sum(pages), 2, hkv, P * D), float("nan"), dtype=torch.bfloat16)     # (a key tile [P][D], a value tile [D][P])
    ks, vs = [], []
    for i, p in enumerate(pos):
        k, v = rand(p + 1, hkv, D, seed=20 + i).bfloat16(), rand(p + 1, hkv, D, seed=160 + i).bfloat16()
        ids = order[at:at + pages[i]]
        at += pages[i]
        table[i, :pages[i]] = ids
        for j in range(pages[i]):
            part = slice(j * P, min(p + 1, (j + 1) * P))
            n = part.stop - part.start
            cache[ids[j], 0].view(hkv, P, D)[:, :n] = k[part].transpose(0, 1)
            cache[ids[j], 1].view(hkv, D, P)[:, :, :n] = v[part].permute(1, 2, 0)
        ks.append(k)
        vs.append(v)
    return cache.view(-1, 2, hkv, P, D).to(DEV), table.to(DEV), ks, vs


EDGES = [0, 1, 15, 16, 17, 47, 48, 63, 64, 511, 512, 513, 800, 1023]
# nine tokens and sixteen (with up to four key/value heads splits, else segments of 512 keys), seventeen and more (splits for one head; one
# segment up to 1024 positions, and up to 2048 with many heads; else segments of 512)
MANY = {"nine": EDGES[5:], "sixteen": EDGES + [1024, 1100], "sixteen far": [127, 128, 511, 512, 767, 768, 769, 895, 896, 1023, 1024, 1535, 1536, 1537, 2047, 2600],
        "few": EDGES[:8] + [301, 302, 303, 304, 305, 306, 307, 1000, 1008, 1023], "seventeen": EDGES + [1024, 1100, 1535], "cut": EDGES + [1536, 2100, 2101, 300, 301, 302],
        "long": EDGES + [4300] + [33] * 185}


@pytest.mark.parametrize("hq,hkv,D,P", [(8, 4, 128, 16), (16, 1, 128, 48), (6, 2, 64, 16), (4, 4, 64, 32), (16, 8, 128, 16), (10, 5, 64, 48)])
@pytest.mark.parametrize("which", list(MANY))
def test_a_block_walks_a_tokens_keys(ops, hq, hkv, D, P, which):
    pos = MANY[which]
    n = len(pos)
    cache, table, ks, vs = _requests(pos, hkv, D, P)
    q = rand(n, hq, D, seed=hq).bfloat16()
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device=DEV)
    scale = 1.5 / D ** 0.5
    seen = dict(dec_tokens=i32(range(n)), max_dec_position=max(pos), dec_blocks=True)
    out = ops.attention(q.to(DEV), cache, i32(pos), i32(range(n)), table, scale, **seen).cpu()
    qkv = torch.stack([torch.cat([q[i].flatten(), ks[i][-1].flatten(), vs[i][-1].flatten()]) for i in range(n)])
    # (the new key and value are written where they already lie: unwritten for it)
    slots = [int(table[i, p // P]) * P + p % P for i, p in enumerate(pos)]
    fresh = cache.clone()
    for s in slots:
        fresh[s // P, 0, :, s % P] = float("nan")
        fresh[s // P, 1].view(hkv, D, P)[:, :, s % P] = float("nan")
    fused = ops.attention_decode_fused(qkv.to(DEV), hq, fresh, i32(pos), i32(range(n)), table, scale, 0, None, max(pos), None, None, 1e-6,
                                       None, i32(slots), dec_blocks=True).cpu()
    assert torch.equal(torch.nan_to_num(fresh.float()), torch.nan_to_num(cache.float()))
    for i, p in enumerate(pos):
        k, v = ks[i].double(), vs[i].double()
        w = torch.softmax(torch.stack([k[:, h * hkv // hq] @ q[i, h].double() for h in range(hq)]) * scale, -1)
        want = torch.stack([w[h] @ v[:, h * hkv // hq] for h in range(hq)])
        # (the weights and the result are rounded to bfloat16: 2^-9 of each weight times its value, and of the result)
        bound = 2.0 ** -8 * (torch.stack([w[h] @ v[:, h * hkv // hq].abs() for h in range(hq)]) + want.abs())
        for got in (out, fused):
            assert ((got.view(n, hq, D)[i].double() - want).abs() <= bound).all(), p


@pytest.mark.parametrize("hq,hkv", [(8, 4), (16, 8)])
def test_bits_of_nine_to_sixteen_tokens(ops, hq, hkv):
    """A token's bits are the same beside eight others and beside fifteen, with keys in one segment (written as they are joined) and in several
    (through the merge), and with its rows in another order."""
    D, P = 128, 16
    pos = [5, 100, 300, 400, 500, 511, 64, 17, 250, 700, 1500, 512, 900, 30, 31, 2]
    cache, table, _, _ = _requests(pos, hkv, D, P)
    qkv = rand(len(pos), (hq + 2 * hkv) * D, seed=3).bfloat16().to(DEV)
    qw, kw, turn = 1 + rand(D, seed=1).to(DEV) / 4, 1 + rand(D, seed=2).to(DEV) / 4, rand(2048, D, seed=4).to(DEV)
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device=DEV)

    def run(which, most):
        got = ops.attention_decode_fused(qkv, hq, cache.clone(), i32(pos), i32(range(len(pos))), table, 0.1, 0, i32(which), most, qw, kw, 1e-6,
                                         turn, None, dec_blocks=True)
        return got[which]
    every = run(list(range(16)), 1500)
    assert torch.equal(run(list(range(9)), 511), every[:9])
    assert torch.equal(run(list(range(9)), 4000), every[:9])
    back = list(range(15, 3, -1))
    assert torch.equal(run(back, 1535), every[back])


@pytest.mark.parametrize("n,longest,ends", [(24, 300, (511,)), (24, 700, (1023,)), (40, 1100, (1535, 2047)), (17, 1700, (2047,)), (33, 2100, (2200, 3071))])
def test_bits_of_a_step_as_it_comes_and_recorded(ops, n, longest, ends):
    """More than sixteen tokens: a recorded step knows the end of the stretch that the last position lies in, another the position."""
    hq, hkv, D, P = 16, 8, 128, 16
    pos = [longest] + [(97 * i) % longest for i in range(1, n)]
    cache, table, _, _ = _requests(pos, hkv, D, P)
    q, i32 = rand(n, hq, D, seed=1).bfloat16().to(DEV), lambda x: torch.tensor(x, dtype=torch.int32, device=DEV)
    run = lambda most: ops.attention(q, cache, i32(pos), i32(range(n)), table, 0.1, dec_tokens=i32(range(n)), max_dec_position=most, dec_blocks=True)
    want = run(longest)
    for end in ends:
        assert torch.equal(run(end), want), end


@pytest.mark.parametrize("hq,hkv,rows", [(8, 4, 1), (8, 4, 70), (8, 1, 200), (6, 2, 33)])
@pytest.mark.parametrize("singles", [1, 15, 40])
def test_single_tokens_beside_a_portion_in_one_launch(ops, hq, hkv, rows, singles):
    """Single tokens as groups of one row of the prefill kernel, beside a portion's rows: what the decode and the prefill kernel compute apart,
    with the tiles from the host and made on the device."""
    from qwen_engine_amd.parts.attention import prefill_tiles
    D, P, behind = 128, 16, 45
    pos = [(i * 37) % 600 for i in range(singles)]
    cache, table, _, _ = _requests(pos + [behind + rows - 1], hkv, D, P)
    T, R = singles + rows, ops.prefill_tile_rows(hq, hkv)
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device=DEV)
    positions, seq = i32(pos + list(range(behind, behind + rows))), i32(list(range(singles)) + [singles] * rows)
    q = rand(T, hq, D, seed=5).bfloat16().to(DEV)
    scale = 1.5 / D ** 0.5
    apart = ops.attention(q, cache, positions, seq, table, scale, dec_tokens=i32(range(singles)), max_dec_position=max(pos),
                          other_tokens=i32(range(singles, T)), other_tiles=i32(prefill_tiles([(singles, rows)], R)).view(-1, 2))
    flat = prefill_tiles([(i, 1) for i in range(singles)] + [(singles, rows)], R)
    tiles = ops.prefill_tiles_on_device(i32([[singles, 0], [singles, rows]]), R, -(-rows // (4 * R)) + 1, singles)
    assert tiles.cpu().flatten().tolist()[:len(flat)] == flat and tiles[len(flat) // 2:, 1].cpu().tolist() == [0] * 4
    together = [ops.attention(q, cache, positions, seq, table, scale, other_tokens=i32(range(T)), other_tiles=t)
                for t in (tiles, i32(flat).view(-1, 2))]
    assert torch.equal(together[0], together[1])
    # (weights and results are rounded to bfloat16 on both sides, at other references: 2^-8 of values of order one, weighed)
    assert (together[0].float() - apart.float()).abs().max() <= 2.0 ** -7 * 4
    assert float((together[0].float() - apart.float()).norm() / apart.float().norm()) < 2.0 ** -8
    if rows > 1 and hq // hkv in (1, 2, 4, 8):
        assert torch.equal(together[0][singles:], apart[singles:])


@pytest.mark.parametrize("wide", [1.0, 4.0])
@pytest.mark.parametrize("singles,keys", [(15, 300), (40, 600)])
def test_single_tokens_beside_a_portion_err_as_by_themselves(ops, singles, keys, wide):
    """Against 64 bits, in the mean of six inputs, hardly more than what the decode kernel gives.  An error is the weights' rounding, but for each walk's
    largest, which is 1: the decode kernel has a walk for every 128 keys.  Of 128 keys with scores of spread 1 the largest weight's square, about e^(2 * 2.5),
    is a sixth of the squares' sum, 128 e^2: one exact weight in 600 keys instead of five errs by a twelfth at the most more."""
    from qwen_engine_amd.parts.attention import prefill_tiles
    hq, hkv, D, P, rows = 16, 8, 128, 16, 20
    R, i32 = ops.prefill_tile_rows(hq, hkv), lambda x: torch.tensor(x, dtype=torch.int32, device=DEV)
    apart = together = 0.0
    for seed in range(6):
        pos = [(keys // 2 + (i + seed) * 37) % keys for i in range(singles)]
        cache, table, ks, vs = _requests(pos + [rows - 1], hkv, D, P)
        T, scale = singles + rows, wide * D ** -0.5
        q = rand(T, hq, D, seed=seed).bfloat16()
        positions, seq = i32(pos + list(range(rows))), i32(list(range(singles)) + [singles] * rows)
        flat = prefill_tiles([(i, 1) for i in range(singles)] + [(singles, rows)], R)
        one = ops.attention(q.to(DEV), cache, positions, seq, table, scale, other_tokens=i32(range(T)), other_tiles=i32(flat).view(-1, 2),
                            prefill_singles=singles)
        two = ops.attention(q.to(DEV), cache, positions, seq, table, scale, dec_tokens=i32(range(singles)), max_dec_position=max(pos))
        for i in range(singles):
            k, v = ks[i].double(), vs[i].double()
            w = torch.softmax(torch.stack([k[:, h * hkv // hq] @ q[i, h].double() for h in range(hq)]) * scale, -1)
            want = torch.stack([w[h] @ v[:, h * hkv // hq] for h in range(hq)])
            together += float((one[i].cpu().double() - want).norm() / want.norm())
            apart += float((two[i].cpu().double() - want).norm() / want.norm())
    assert together <= 13 / 12 * apart


def test_recorded_steps_choose_as_steps_that_run_as_they_come(ops):
    """Single tokens beside a portion: in one launch or two does not hang on what a recorded step fills up."""
    from qwen_engine_amd.engine import ModelRunner
    from qwen_engine_amd.parts.attention import PagedAttention
    step = ModelRunner.MIXED_GRAPH_STEP
    for n in (1, 2, 7, 8, 9, 15, 33, 50, 70, 97, 101):
        for last in (0, 300, 511, 512, 700, 1023, 1024, 1500):
            end = PagedAttention.graph_key(last) * ops.DECODE_SPLIT_KEYS - 1
            for rows in (2, 100, 127, 128, 129, 200, 255, 256, 257, 500):
                for keys in (rows, 1024, 1025, 3000):
                    for heads in (1, 2, 4, 8, 16):
                        comes = ops.prefill_takes_single(n, last, rows, keys, heads)
                        then = ops.prefill_takes_single(ModelRunner.graph_rows(n), end, -(-rows // step) * step, keys, heads)
                        assert comes == then, (n, last, rows, keys, heads)


def test_few_walks_beside_few_rows_go_apart(ops):
    """Beyond 512 positions one block's walk decides, which was up to a fifth slower than splits and the portion by itself."""
    for n, heads in ((8, 1), (8, 4), (8, 8), (15, 1), (15, 4), (33, 2)):
        assert not ops.prefill_takes_single(n, 960, 64, 64, heads) and ops.prefill_takes_single(n, 960, 400, 400, heads)
        assert ops.prefill_takes_single(n, 500, 64, 64, heads)
    assert ops.prefill_takes_single(15, 960, 64, 64, 8) and ops.prefill_takes_single(33, 960, 64, 64, 4) and not ops.prefill_takes_single(15, 1024, 64, 64, 8)


def test_where_the_step_before_goes_inside(ops):
    """Up to 64 rows of either type."""
    asked = lambda n, dtype: ops.attention_decode_fused_preferred(torch.empty(n, 8, dtype=dtype, device=DEV))
    for dtype in (torch.bfloat16, torch.float32):
        assert all(asked(n, dtype) for n in (1, 16, 17, 24, 48, 64)) and not asked(65, dtype)


@pytest.mark.parametrize("n,hkv,keys", [(9, 1, 680), (12, 2, 1000), (24, 1, 680), (20, 8, 3000)])
def test_blocks_only_where_they_are_not_slower(ops, n, hkv, keys):
    """With splits of 128 keys beside it: a sixth more time at the most (with a block's walk of 512 or 1024 keys each on a nearly idle chip it was 1.34 to
    1.47 times)."""
    hq, D, P = 2 * hkv, 128, 16
    pos = [keys // 2 + keys * i // (n - 1) for i in range(n)]
    per = max(pos) // P + 1
    cache = torch.zeros(n * per, 2, hkv, P, D, dtype=torch.bfloat16, device=DEV)
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device=DEV)
    table, end = torch.arange(n * per, dtype=torch.int32, device=DEV).view(n, per), max(pos) | 1023
    qkv = torch.zeros(n, (hq + 2 * hkv) * D, dtype=torch.bfloat16, device=DEV)
    positions, seq = i32(pos), i32(range(n))

    def recorded(blocks):
        run = lambda: ops.attention_decode_fused(qkv, hq, cache, positions, seq, table, 0.1, 0, None, end, None, None, 1e-6, None, None, dec_blocks=blocks)
        run()
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            for _ in range(20):
                run()
        return graph

    def took(graph):
        a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        a.record()
        graph.replay()
        b.record()
        b.synchronize()
        return a.elapsed_time(b)
    one, two = recorded(True), recorded(False)
    times = [(took(one), took(two)) for _ in range(8)]
    assert min(t[0] for t in times) < 7 / 6 * min(t[1] for t in times)


@pytest.mark.parametrize("T,H,n", [(1, 8, 2), (3, 100, 300), (9, 1024, 1), (2, 1030, 700)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_embedding_with_a_block_tables_updates(ops, T, H, n, dtype):
    """The rows, and the table's entries as scatter_int writes them, in one launch; rows at odd addresses."""
    emb = rand(50, H + 1, seed=1).to(dtype).to(DEV)[:, 1:].contiguous()
    odd = torch.empty(50 * H + 1, dtype=dtype, device=DEV)[1:].view(50, H).copy_(emb)
    ids = torch.randint(0, 50, (T,), generator=torch.Generator().manual_seed(2)).int().to(DEV)
    idx = torch.randperm(4 * n, generator=torch.Generator().manual_seed(3))[:n].int().to(DEV)
    idx[::3] = -1
    val = torch.arange(n, dtype=torch.int32, device=DEV)
    want, got = torch.full((4, n), 7, dtype=torch.int32, device=DEV), torch.full((4, n), 7, dtype=torch.int32, device=DEV)
    ops.scatter_int(want, idx, val)
    for table in (emb, odd):
        assert torch.equal(ops.embedding(ids, table, update=(got, idx, val)), emb[ids.long()].float())
    assert torch.equal(got, want) and torch.equal(ops.embedding(ids, emb), emb[ids.long()].float())


@pytest.mark.parametrize("n", [1, 63, 64, 65, 130])
def test_numbers_that_travel_with_the_launch(ops, n):
    g = torch.Generator().manual_seed(n)
    places, values = torch.randperm(200, generator=g)[:n], torch.randint(-5, 1 << 30, (n,), generator=g)
    table = torch.full((200,), 7, dtype=torch.int32, device=DEV)
    want = table.cpu()
    want[places] = values.int()
    ops.set_ints(table, places.tolist(), values.tolist())
    assert torch.equal(table.cpu(), want)
    with pytest.raises(ops.KernelError):
        ops.set_ints(table, [200], [0])
    assert torch.equal(table.cpu(), want)
