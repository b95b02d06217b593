"""The layers of a step of single new tokens in one launch (``ops.decode_chain``) against the same layers in plain torch: at the
edges of tiles, segments, pages and shares, and with other numbers of blocks than compute units."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
D = 128


@pytest.fixture(scope="module")
def ops():
    from qwen_engine_amd.kernels import ops
    ops.load_library()
    return ops


def make(ops, n, H, Hq, Hkv, I, P, pos, seed=1, norms=True, rope=True):
    """Layers, caches whose pages lie anywhere, and the step's arrays; what no token has written yet is NaN."""
    g = torch.Generator().manual_seed(seed)
    r = lambda *s, std=0.02: torch.randn(*s, generator=g) * std
    T, per = len(pos), max(pos) // P + 1
    perm = torch.randperm(T * per, generator=g).view(T, per) + 1
    layers = []
    for _ in range(n):
        kv = torch.full((T * per + 1, 2, Hkv, P, D), float("nan"), dtype=torch.bfloat16)
        for i, p in enumerate(pos):
            k, v = r(Hkv, per * P, D, std=1.0).bfloat16(), r(Hkv, per * P, D, std=1.0).bfloat16()
            k[:, p:], v[:, p:] = float("nan"), float("nan")
            for j in range(per):                     # keys [P, D], values transposed [D, P]
                kv[perm[i, j], 0] = k[:, j * P:(j + 1) * P]
                kv[perm[i, j], 1] = v[:, j * P:(j + 1) * P].transpose(1, 2).reshape(Hkv, P, D)
        layers.append(dict(w_qkv=r((Hq + 2 * Hkv) * D, H).bfloat16(), w_o=r(H, Hq * D).bfloat16(), w_gate=r(I, H).bfloat16(), w_up=r(I, H).bfloat16(),
                           w_down=r(H, I).bfloat16(), norm1=1 + r(H, std=0.1), norm2=1 + r(H, std=0.1),
                           q_norm=1.4 + r(D, std=0.1) if norms else None, k_norm=1.4 + r(D, std=0.1) if norms else None,
                           eps1=1e-6, eps2=1e-5, cache=kv))
    f = torch.outer(torch.arange(max(pos) + 1).float(), 1e6 ** (-torch.arange(0, D, 2).float() / D))
    table = torch.cat([f.cos(), f.sin()], -1).contiguous() if rope else None
    bt = torch.zeros(T + 1, per, dtype=torch.int32)
    bt[:T] = perm
    slots = torch.tensor([int(perm[i, p // P]) * P + p % P for i, p in enumerate(pos)], dtype=torch.int32)
    return layers, table, bt, slots, perm, r(T, H, std=1.0)


def on_device(ops, layers):
    out = []
    for L in layers:
        d = {k: v.to(DEV) if isinstance(v, torch.Tensor) else v for k, v in L.items() if k not in ("w_gate", "w_up")}
        d["w_gu"] = ops.interleave_gate_up(L["w_gate"], L["w_up"]).to(DEV)
        out.append(d)
    return out


def plain(layers, table, perm, h, pos, Hq, Hkv, P):
    """In 64 bits, with the operands of the products rounded to bfloat16 where the engine rounds them."""
    rd = lambda x: x.bfloat16().double()
    rms = lambda x, eps: x * torch.rsqrt((x * x).mean(-1, keepdim=True) + eps)
    h = h.double()
    T, G, new = h.shape[0], Hq // Hkv, []
    for L in layers:
        qkv = rd(rd(rms(h, L["eps1"]) * L["norm1"].double()) @ L["w_qkv"].double().t()).view(T, Hq + 2 * Hkv, D)
        q, k, v = qkv[:, :Hq], qkv[:, Hq:Hq + Hkv], qkv[:, Hq + Hkv:]
        if L["q_norm"] is not None:
            q, k = rms(q, 1e-6) * L["q_norm"].double(), rms(k, 1e-6) * L["k_norm"].double()
        if table is not None:
            c, s = (table[pos][:, None, i * D // 2:(i + 1) * D // 2].double() for i in (0, 1))
            turn = lambda x: torch.cat([x[..., :D // 2] * c - x[..., D // 2:] * s, x[..., D // 2:] * c + x[..., :D // 2] * s], -1)
            q, k = turn(q), turn(k)
        q, k = rd(q), rd(k)
        new.append((k, v))
        o = torch.empty(T, Hq, D, dtype=torch.float64)
        for t, p in enumerate(pos):
            pages = L["cache"][perm[t, :p // P + 1]].double()
            ks = torch.cat([pages[:, 0].permute(1, 0, 2, 3).reshape(Hkv, -1, D)[:, :p], k[t][:, None]], 1)
            vs = torch.cat([pages[:, 1].reshape(-1, Hkv, D, P).permute(1, 0, 3, 2).reshape(Hkv, -1, D)[:, :p], v[t][:, None]], 1)
            w = torch.softmax((q[t].view(Hkv, G, D) @ ks.transpose(1, 2)) * D ** -0.5, -1)
            o[t] = (w @ vs).reshape(Hq, D)
        h = h + rd(o.reshape(T, -1)) @ L["w_o"].double().t()
        x = rd(rms(h, L["eps2"]) * L["norm2"].double())
        a = x @ L["w_gate"].double().t()
        h = h + rd(a * torch.sigmoid(a) * (x @ L["w_up"].double().t())) @ L["w_down"].double().t()
    return h, new


def check(ops, n, H, Hq, Hkv, I, P, pos, units=0, seed=1, write=True, shared=None, late=None, **kw):
    layers, table, bt, slots, perm, h0 = make(ops, n, H, Hq, Hkv, I, P, pos, seed, **kw)
    want, new = plain(layers, table, perm, h0, pos, Hq, Hkv, P)
    dev = on_device(ops, layers)
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device=DEV)
    args = (i32(pos), i32(list(range(len(pos)))), bt.to(DEV), slots.to(DEV) if write else None, Hq, D ** -0.5, max(pos), 1e-6,
            None if table is None else table.to(DEV), None if shared is None else i32(shared))
    h = h0.to(DEV)
    ops.decode_chain(h, dev, *args, units=units, late=late)
    torch.cuda.synchronize()
    # what the layers add, of which each of some ten roundings to bfloat16 a layer leaves 2^-9 at the most, 2^-10 in the mean square
    err = float((h.cpu().double() - want).norm() / (want - h0.double()).norm())
    assert err < 2.0 ** -9 * (2 * n) ** 0.5 * 3, err
    for L, d, (k, v) in zip(layers, dev, new):
        for t, p in enumerate(pos):
            page, at = int(perm[t, p // P]), p % P
            got_k, got_v = d["cache"][page, 0, :, at].cpu(), d["cache"][page, 1].reshape(Hkv, D, P)[:, :, at].cpu()
            if write:                                # (a rounding of the key may fall the other way)
                assert float((got_k.double() - k[t]).norm() / k[t].norm()) < 2.0 ** -7
                assert float((got_v.double() - v[t]).norm() / v[t].norm()) < 2.0 ** -7
                d["cache"][page, 0, :, at] = float("nan")
                d["cache"][page, 1].view(Hkv, D, P)[:, :, at] = float("nan")
        same = d["cache"].cpu().view(torch.int16) == L["cache"].view(torch.int16)
        assert bool((same | (torch.isnan(d["cache"].cpu()) & torch.isnan(L["cache"]))).all())       # nothing else was written
    return h, dev, args, h0


@pytest.mark.parametrize("pos", [[0], [1, 15], [16, 17, 47], [63, 64, 65, 0], [127, 128, 129, 5, 900], [2047, 2048, 3, 511, 512, 513, 0, 2111]])
@pytest.mark.parametrize("Hq,Hkv,P", [(2, 2, 16), (8, 1, 32), (4, 2, 64)])
def test_edges_of_tiles_segments_and_pages(ops, pos, Hq, Hkv, P):
    check(ops, 2, 256, Hq, Hkv, 384, P, pos, seed=len(pos) + P)


@pytest.mark.parametrize("H,Hq,Hkv,I,rows", [(128, 1, 1, 128, 1), (1024, 16, 8, 3072, 8), (1152, 9, 3, 2048, 3), (2048, 16, 8, 6144, 6), (2176, 8, 8, 640, 4),
                                             (4096, 32, 8, 12288, 1), (2560, 32, 8, 9728, 2), (2560, 32, 8, 9728, 4), (5120, 40, 8, 17408, 1), (1024, 4, 4, 12800, 3),
                                             (4096, 32, 8, 12288, 3)])
def test_widths(ops, H, Hq, Hkv, I, rows):
    """Products whose chunks of K do not come out even, shares that differ from block to block, both sizes of the rings."""
    assert ops.decode_chain_supported(rows, H, Hq, Hkv, D, I, 16)
    check(ops, 1, H, Hq, Hkv, I, 16, [50 + 77 * i for i in range(rows)], seed=H)


@pytest.mark.parametrize("units", [1, 2, 3, 37, 255])
def test_any_number_of_blocks(ops, units):
    """What is left to fewer blocks than there are compute units: several units of the attention and rounds of a product a block, more tiles a
    wave than shared memory holds."""
    check(ops, 2, 512, 4, 2, 768, 16, [700, 33, 4100 if units < 3 else 0], units=units)


def test_many_tiles_of_a_wave(ops):
    check(ops, 2, 256, 8, 8, 256, 64, [11000, 3, 9999], units=40)


def test_without_norms_rotation_or_a_place_to_write(ops):
    check(ops, 2, 256, 4, 2, 384, 16, [40, 3], norms=False)
    check(ops, 2, 256, 4, 2, 384, 16, [40, 3], rope=False)
    check(ops, 2, 256, 4, 2, 384, 16, [40, 3], write=False)
    check(ops, 2, 256, 4, 2, 384, 16, [300, 200], shared=[256, 0, 0])


def test_more_layers_than_a_launch_holds(ops):
    n = ops.load_library().qe_decode_chain_layers() + 3
    check(ops, n, 128, 1, 1, 128, 16, [20, 5])


def test_the_same_bits_again_recorded_and_on_two_streams(ops):
    """A result does not depend on the run: launches beside each other on two streams (each with the blocks that find a place) and
    replays with other work between them."""
    h, dev, args, h0 = check(ops, 4, 1024, 16, 8, 3072, 16, [600, 20, 1500])
    for d, L in zip(dev, make(ops, 4, 1024, 16, 8, 3072, 16, [600, 20, 1500])[0]):
        d["cache"].copy_(L["cache"])
    runs = []
    streams = [torch.cuda.Stream(), torch.cuda.Stream()]
    copies = [[dict(d, cache=d["cache"].clone()) for d in dev] for _ in streams]
    torch.cuda.synchronize()
    for _ in range(10):
        for s, layers in zip(streams, copies):
            with torch.cuda.stream(s):
                x = h0.to(DEV, non_blocking=False)
                ops.decode_chain(x, layers, *args)
                runs.append(x)
    torch.cuda.synchronize()
    assert all(torch.equal(x, h) for x in runs)
    graph, static = torch.cuda.CUDAGraph(), h0.to(DEV)
    with torch.cuda.stream(streams[0]):
        ops.decode_chain(static, dev, *args)
    torch.cuda.synchronize()
    with torch.cuda.graph(graph, stream=streams[0]):
        ops.decode_chain(static, dev, *args)
    for _ in range(4):
        static.copy_(h0)
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(static, h)
        torch.ones(1 << 20, device=DEV).sum().item()


@pytest.mark.parametrize("H,Hq,Hkv,I", [(256, 4, 2, 384), (1024, 16, 8, 1024)])
def test_a_token_alone_and_in_company(ops, H, Hq, Hkv, I):
    """A row's bits, and those of the key and value it writes, follow neither the rows beside it nor the number of blocks: positions at
    both sides of where the segments' length changes, and rows whose units are dealt to one block and to many."""
    pos = [2559, 0, 130, 8191, 700, 2560, 8192, 16500]
    layers, table, bt, slots, perm, h0 = make(ops, 2, H, Hq, Hkv, I, 16, pos, seed=9)
    fresh = on_device(ops, layers)
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device=DEV)
    bt, table = bt.to(DEV), table.to(DEV)

    def run(rows, units=0):
        dev = [dict(d, cache=d["cache"].clone()) for d in fresh]
        h = h0[rows].to(DEV)
        ops.decode_chain(h, dev, i32([pos[r] for r in rows]), i32(rows), bt, slots[rows].to(DEV), Hq, D ** -0.5, max(pos[r] for r in rows), 1e-6, table, units=units)
        new = [torch.stack([d["cache"][int(perm[r, pos[r] // 16]), 0, :, pos[r] % 16] for d in dev]) for r in rows]
        return h.cpu(), [x.cpu() for x in new]

    want_h, want_k = run(list(range(8)))
    assert bool(torch.isfinite(want_h).all())
    for rows in ([0], [1], [3], [7], [6, 2], [5, 0], [4, 1, 7], [2, 3, 5, 6], [7, 6, 5, 4, 3]):
        for units in (0, 11):
            h, k = run(rows, units)
            for i, r in enumerate(rows):
                assert torch.equal(h[i], want_h[r]) and torch.equal(k[i], want_k[r]), (rows, r, units)


@pytest.mark.parametrize("rows", [1, 3, 8])
def test_a_wait_in_vain_ends_and_is_told(ops, rows):
    """Blocks that have work and do not come: every wait ends, the rows are NaN, the word is set; the next launch knows nothing of it."""
    pos = [40 + 150 * i for i in range(rows)]
    late = torch.zeros(1, dtype=torch.int32).pin_memory()
    h, dev, args, h0 = check(ops, 2, 512, 4, 2, 768, 16, pos, late=late)
    assert int(late) == 0
    x = h0.to(DEV)
    ops.decode_chain(x, [dict(d, cache=d["cache"].clone()) for d in dev], *args, late=late, limit_us=3000, absent=2)
    torch.cuda.synchronize()
    assert int(late) == 1 and bool(torch.isnan(x).any(1).all())
    late.zero_()
    y = h0.to(DEV)
    dev = on_device(ops, make(ops, 2, 512, 4, 2, 768, 16, pos)[0])
    ops.decode_chain(y, dev, *args, late=late, limit_us=3000)
    torch.cuda.synchronize()
    assert int(late) == 0 and torch.equal(y, h)
    with pytest.raises(ops.KernelError):
        ops.decode_chain(y, dev, *args, late=torch.zeros(1, dtype=torch.int32))


def test_beside_a_product_that_holds_half_of_the_chip(ops):
    """Which blocks take part is settled for the whole step: one that begins while others hold the units waits for them instead of going
    through all its layers with the few that are free (which took seven times as long as all)."""
    pos = [2000] * 8
    layers, table, bt, slots, perm, h0 = make(ops, 1, 1024, 16, 8, 3072, 16, pos)
    dev = on_device(ops, layers) * 12
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device=DEV)
    args = (i32(pos), i32(list(range(8))), bt.to(DEV), slots.to(DEV), 16, D ** -0.5, 2000, 1e-6, table.to(DEV))
    x, w = torch.ones(1280, 49152, dtype=torch.bfloat16, device=DEV), torch.ones(6144, 49152, dtype=torch.bfloat16, device=DEV)
    y, h = torch.empty(1280, 6144, dtype=torch.bfloat16, device=DEV), h0.to(DEV)
    streams = [torch.cuda.Stream(), torch.cuda.Stream()]

    def timed(stream, f):
        begin, end = (torch.cuda.Event(enable_timing=True) for _ in range(2))
        with torch.cuda.stream(stream):
            begin.record()
            f()
            end.record()
        return begin, end

    beside, alone, product = [], [], []
    for _ in range(4):
        torch.cuda.synchronize()
        a = timed(streams[0], lambda: ops.decode_chain(h, dev, *args))
        torch.cuda.synchronize()
        b = timed(streams[1], lambda: ops.gemm(x, w, out=y))
        c = timed(streams[0], lambda: ops.decode_chain(h, dev, *args))
        torch.cuda.synchronize()
        for times, (begin, end) in zip((alone, product, beside), (a, b, c)):
            times.append(begin.elapsed_time(end))
    # (as soon as the product is done, and then as long as alone: 0.73, 0.55 and 1.2 ms)
    assert min(beside) < min(product) + 3 * min(alone), (beside, product, alone)


def test_refuses_what_it_does_not_take(ops):
    assert not ops.decode_chain_supported(9, 1024, 16, 8, 128, 3072, 16)          # rows
    assert not ops.decode_chain_supported(1, 1024, 16, 8, 64, 3072, 16)           # head size
    assert not ops.decode_chain_supported(1, 1000, 16, 8, 128, 3072, 16)          # width
    assert not ops.decode_chain_supported(1, 1024, 16, 8, 128, 3000, 16)
    assert not ops.decode_chain_supported(1, 1024, 16, 1, 128, 3072, 16)          # queries to a key
    assert not ops.decode_chain_supported(1, 1024, 16, 8, 128, 3072, 48)          # page
    assert not ops.decode_chain_supported(6, 4096, 32, 8, 128, 12288, 16)         # shared memory
    assert ops.decode_chain_supported(3, 4096, 32, 8, 128, 12288, 16) and not ops.decode_chain_preferred(3, 4096, 32, 8, 128, 12288, 16)
    assert ops.decode_chain_supported(1, 5120, 64, 8, 128, 25600, 16) and not ops.decode_chain_preferred(1, 5120, 64, 8, 128, 25600, 16)
    layers, table, bt, slots, perm, h0 = make(ops, 1, 256, 2, 1, 384, 16, [5])
    dev = on_device(ops, layers)
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device=DEV)
    with pytest.raises(ops.KernelError):
        ops.decode_chain(h0.to(DEV), dev, i32([5, 6]), i32([0]), bt.to(DEV), None, 2, 0.1, 5)
    with pytest.raises(ops.KernelError):
        ops.decode_chain(h0.to(DEV), [dict(dev[0], w_o=dev[0]["w_o"].float())], i32([5]), i32([0]), bt.to(DEV), None, 2, 0.1, 5)
    with pytest.raises(ops.KernelError):
        ops.decode_chain(h0.to(DEV), [dict(dev[0], k_norm=None)], i32([5]), i32([0]), bt.to(DEV), None, 2, 0.1, 5)


@pytest.mark.parametrize("rows,H,Hq,Hkv,I,position,quicker", [
    # rings of eight kilobytes: many rows, a wide middle, seven or eight queries to a key
    (3, 2304, 16, 8, 9216, 200, True), (3, 2560, 32, 8, 9728, 200, False), (4, 3072, 24, 3, 8192, 200, False), (4, 2560, 32, 8, 9728, 32000, False),
    (3, 3072, 24, 8, 12288, 32000, False), (6, 2048, 16, 8, 6144, 200, True),
    (2, 3072, 28, 4, 12288, 200, True), (1, 3584, 28, 4, 18944, 200, False), (2, 4096, 32, 8, 16384, 200, True), (2, 5120, 40, 8, 14592, 200, False),
    (1, 4224, 32, 4, 12288, 200, False), (2, 5120, 48, 6, 12288, 200, False), (2, 3584, 28, 7, 18944, 200, False),
    # of twelve
    (1, 3584, 28, 7, 18944, 200, True), (2, 5120, 40, 8, 13824, 200, True), (3, 3072, 24, 8, 8192, 200, True), (2, 4096, 32, 8, 12288, 40000, True),
    # one request with one key/value head
    (1, 1024, 8, 1, 3072, 45000, True), (1, 1024, 8, 1, 3072, 60000, False), (1, 1024, 4, 1, 3072, 60000, False), (2, 1024, 8, 1, 3072, 120000, True),
    (1, 1024, 16, 2, 3072, 120000, True), (1, 2048, 8, 1, 6144, 60000, True), (1, 2048, 8, 1, 6144, 120000, False)])
def test_where_it_is_the_quicker_way(ops, rows, H, Hq, Hkv, I, position, quicker):
    """Both sides of every line of the rule, at sizes where both ways were measured."""
    assert ops.decode_chain_preferred(rows, H, Hq, Hkv, 128, I, 16, position) == quicker
