"""Forms of the kernels that are chosen by sizes: each at the edges of its range against the plain product or mechanism in
64 bits, and against the other forms."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.fixture(scope="module")
def ops():
    from qwen_engine_amd.kernels import ops
    ops.load_library()
    return ops


def rand(*shape, seed=0, dtype=torch.float32, scale=1.0):
    g = torch.Generator().manual_seed(seed)
    return (torch.randn(*shape, generator=g) * scale).to(dtype)


@pytest.mark.parametrize("M", [1, 4, 5, 16, 17, 33, 64, 65, 130, 700])
@pytest.mark.parametrize("N,K", [(17, 3), (64, 15), (33, 16), (100, 250), (1024, 257), (40, 1008), (6160, 272), (1040, 4100)])
def test_float32_gemm_sums_in_one_order(ops, M, N, K):
    """The float32 product by rows and by tiles (the number of rows and of tiles decides): against the 64-bit product, and
    every row the same bits whatever kernel takes it; operands that lie at odd addresses give the same bits too."""
    x, w = rand(M, K, seed=1300 + K), rand(N, K, seed=1301 + N)
    want = x.double() @ w.double().t()
    got = ops.gemm(x.to(DEV), w.to(DEV))
    # (a sum of K products rounded K times: at most K u |x| |w|, some sqrt(K) u of it in practice)
    bound = 2.0 ** -24 * 2 * K ** 0.5 * (x.double().abs() @ w.double().abs().t())
    assert ((got.cpu().double() - want).abs() <= bound + 1e-30).all()
    for m in {0, M // 2, M - 1}:
        assert torch.equal(ops.gemm(x[m:m + 1].to(DEV), w.to(DEV))[0], got[m])
    odd = torch.empty(M * K + 1, device=DEV)[1:].view(M, K).copy_(x)
    assert torch.equal(ops.gemm(odd, w.to(DEV)), got)


@pytest.mark.parametrize("M,N,K", [(1, 24, 4), (70, 300, 77), (333, 1023, 1001), (5, 6160, 1020), (20, 40, 36), (64, 1040, 100), (333, 1024, 1000),
                                   (40, 130, 5), (3, 20, 6), (200, 70, 7), (33, 1000, 63), (33, 1000, 65), (520, 2048, 511), (520, 1024, 515),
                                   (744, 640, 20), (2049, 1024, 44)])
def test_float32_gemm_of_rows_that_end_inside_a_step(ops, M, N, K):
    """K a multiple of 4 and no multiple of 16, and neither: by rows and by tiles, one and four groups; what lies behind a row
    (the next one, or nothing) has no part in it, and a view that begins anywhere gives the same bits."""
    x, w = rand(M, K, seed=K), rand(N, K, seed=K + 1)
    want = x.double() @ w.double().t()
    got = ops.gemm(x.to(DEV), w.to(DEV))
    bound = 2.0 ** -24 * 2 * K ** 0.5 * (x.double().abs() @ w.double().abs().t())      # (K products, rounded K times)
    assert ((got.cpu().double() - want).abs() <= bound + 1e-30).all()
    wide = torch.full((M * K + 7,), float("nan"), device=DEV)
    wide[3:3 + M * K] = x.flatten().to(DEV)
    wide_w = torch.full((N * K + 7,), float("nan"), device=DEV)
    wide_w[1:1 + N * K] = w.flatten().to(DEV)
    assert torch.equal(ops.gemm(wide[3:3 + M * K].view(M, K), wide_w[1:1 + N * K].view(N, K)), got)
    assert torch.equal(ops.gemm(x[M // 2:M // 2 + 1].to(DEV), w.to(DEV))[0], got[M // 2])


@pytest.mark.parametrize("tile", [64, 128, 256, 512])
@pytest.mark.parametrize("M,N", [(64 * 5, 128 * 13), (64 * 9 + 1, 128 * 7 + 64), (128 * 11 - 3, 128 * 5), (2300, 640), (130, 128 * 257 + 8)])
def test_tiled_gemm_covers_every_tile(ops, tile, M, N):
    """The walk through the tiles: numbers of tile rows and columns that are no multiples of eight, one band of tile rows and
    several, a last band of one tile row; every sum is a whole number far below 2^24, so the results are exact."""
    if tile >= 256 and M <= 128:
        pytest.skip("no such tile for so few rows")
    g = torch.Generator().manual_seed(M + N)
    K = 192
    x = torch.randint(-3, 4, (M, K), generator=g).bfloat16()
    w = torch.randint(-3, 4, (N, K), generator=g).bfloat16()
    want = (x.float() @ w.float().t()).to(DEV)
    assert torch.equal(ops.gemm(x.to(DEV), w.to(DEV), out_dtype=torch.float32, algo=ops.ALGO_TILE + tile), want)
    parts = ops.gemm(x.to(DEV), w.to(DEV), epilogue=ops.EPI_PARTIAL, splits=3, algo=ops.ALGO_TILE + tile)
    assert torch.equal(parts[0] + parts[1] + parts[2], want)


@pytest.mark.parametrize("M,N,K", [(65, 1024, 1024), (80, 5120, 6400), (144, 256, 4096), (272, 640, 12288), (400, 1024, 2048), (528, 136, 3080),
                                   (1300, 512, 2048), (2049, 1024, 1032)])
def test_branch_products_in_as_many_cuts_as_asked_for(ops, M, N, K):
    """The number of cuts that is asked for leaves every part some of K, is one the product takes, and its parts add up to
    it, whole numbers far below 2^24 exactly."""
    g = torch.Generator().manual_seed(M)
    x = torch.randint(-3, 4, (M, K), generator=g).bfloat16().to(DEV)
    w = torch.randint(-3, 4, (N, K), generator=g).bfloat16().to(DEV)
    splits = ops.gemm_branch_splits(x, w)
    got = ops.gemm(x, w, epilogue=ops.EPI_PARTIAL, splits=splits) if splits else ops.gemm(x, w, out_dtype=torch.float32)[None]
    assert splits in range(7) and len(got) == max(splits, 1)
    assert torch.equal(got.sum(0), x.float() @ w.float().t())


def latent_rows(before, rows, R, dr, page, seed):
    """Requests with ``before`` cached tokens and ``rows`` new ones over scattered pages: (cache, table, positions, tok_seq, the
    requests' rows [keys, R + dr])."""
    keys = [b + n for b, n in zip(before, rows)]
    pages = [-(-k // page) for k in keys]
    order = torch.randperm(sum(pages), generator=torch.Generator().manual_seed(seed))
    cache = torch.full((sum(pages), 1, 1, page, R + dr), float("nan"))       # (what was never written must not be used)
    table = torch.full((len(keys), max(pages)), -1, dtype=torch.int32)
    own, at = [], 0
    for i, k in enumerate(keys):
        c = rand(k, R + dr, seed=seed + 1 + i).bfloat16().float()
        ids = order[at:at + pages[i]]
        at += pages[i]
        table[i, :pages[i]] = ids.int()
        flat = torch.full((pages[i] * page, R + dr), float("nan"))
        flat[:k] = c
        cache[ids, 0, 0] = flat.view(pages[i], page, R + dr)
        own.append(c.double())
    pos = torch.cat([torch.arange(b, b + n) for b, n in zip(before, rows)]).int()
    seq = torch.cat([torch.full((n,), i) for i, n in enumerate(rows)]).int()
    return cache.bfloat16().to(DEV), table.to(DEV), pos.to(DEV), seq.to(DEV), own


@pytest.mark.parametrize("R,dn,dr,dv", [(512, 128, 64, 128), (128, 64, 32, 64), (64, 128, 0, 128), (72, 64, 0, 64), (256, 96, 32, 64)])
@pytest.mark.parametrize("before,rows", [((0,), (1,)), ((0, 0), (33, 130)), ((70, 0, 5), (31, 128, 64)), ((300,), (257,)), ((1000, 3), (5, 700))])
@pytest.mark.parametrize("window,sink,gated", [(0, False, 0), (40, True, 1), (64, False, 2)])
def test_latent_attention_of_portions_with_expanded_keys(ops, R, dn, dr, dv, before, rows, window, sink, gated):
    """Every size of head that the kernel takes, portions that end inside a tile of rows, of keys and of 64 places, windows that
    begin anywhere, against 64-bit attention; the kernel with folded maps beside it."""
    from qwen_engine_amd.parts.attention import prefill_tiles
    H, page, scale, T = 3, 16, 0.11, sum(rows)
    cache, table, pos, seq, own = latent_rows(before, rows, R, dr, page, 17)
    uk, uv = rand(H * dn, R, seed=3, scale=R ** -0.5).bfloat16(), rand(H * dv, R, seed=4, scale=R ** -0.5).bfloat16()
    q = rand(T, H, dn + dr, seed=5, scale=1.5).bfloat16()
    sinks = rand(H, seed=6).to(DEV) if sink else None
    gate = rand(T, H * dv if gated == 1 else H, seed=7).bfloat16().to(DEV) if gated else None
    portions, owner, tiles, group, at = [], [], [], [], 0
    for i, (b, n) in enumerate(zip(before, rows)):
        keys = b + n - (max(0, b - window + 1) if window else 0)
        portions += [at, n, 64 * len(owner)]
        owner += [i] * -(-keys // 64)
        mine = prefill_tiles([(at, n)], 32)
        tiles += mine
        group += [i] * (len(mine) // 8)
        at += n
    i32 = lambda v, *shape: torch.tensor(v, dtype=torch.int32, device=DEV).view(*shape)
    portions = i32(portions, -1, 3)
    ck, kr = ops.latent_gather(cache, pos, seq, table, portions, i32(owner, -1), R, window=window)
    out = torch.full((T, H, dv), float("nan"), dtype=torch.bfloat16, device=DEV)
    ops.latent_prefill(q.to(DEV), ops.gemm(ck, uk.to(DEV)), kr, ops.gemm(uv.to(DEV), ck), out, i32(tiles, -1, 2), i32(group, -1),
                       portions, pos, scale, window=window, sink=sinks, gate=gate)
    qp = torch.empty(T, H, R + dr, dtype=torch.bfloat16, device=DEV)
    qp[..., R:] = q.to(DEV)[..., dn:]
    ops.gemm_heads(q.to(DEV), uk.view(H, dn, R).transpose(1, 2).contiguous().to(DEV), qp)
    folded = torch.empty_like(out)
    ops.gemm_heads(ops.latent_attention(qp, cache, pos, seq, table, R, scale, window=window, sink=sinks),
                   uv.view(H, dv, R).to(DEV), folded, gate)
    want, at = [], 0
    for i, (b, n) in enumerate(zip(before, rows)):
        c = own[i]
        k = torch.cat([(c[:, :R] @ uk.double().t()).view(-1, H, dn), c[:, None, R:].expand(-1, H, dr)], dim=2)
        v = (c[:, :R] @ uv.double().t()).view(-1, H, dv)
        s = torch.einsum("thd,khd->htk", q[at:at + n].double(), k) * scale
        d = torch.arange(b, b + n)[:, None] - torch.arange(b + n)[None, :]
        s = s.masked_fill((d < 0) | ((d >= window) if window else False), float("-inf"))
        if sink:
            s = torch.cat([s, sinks.cpu().double().view(H, 1, 1).expand(H, n, 1)], dim=2)
        p = torch.softmax(s, dim=-1)[..., :b + n]
        want.append(torch.einsum("htk,khd->thd", p, v))
        at += n
    want = torch.cat(want)
    if gated:
        want = want * torch.sigmoid(gate.cpu().double().view(T, H, -1))
    off = lambda t: float((t.cpu().double() - want).norm() / want.norm())
    # keys, values, weights and the result are rounded to bfloat16 once each: 2^-9 / sqrt(3) of the size apiece, the keys'
    # by way of scores of a few units (the folded maps round queries, weights, latent sums and the result)
    print(f"expanded {off(out):.2e} folded {off(folded):.2e}")
    assert off(out) < 5e-3, (off(out), off(folded))


def rms_of(x):
    return x / (x.square().mean(-1, keepdim=True) + 1e-5).sqrt()


@pytest.mark.parametrize("M,N,K", [(1, 24, 128), (8, 4096, 1024), (16, 1000, 512), (17, 256, 64), (65, 192, 136), (300, 1160, 256),
                                   (1100, 2304, 128)])
def test_gelu_in_the_product(ops, M, N, K):
    """The gelu on a product's 32-bit sums, by the kernel for few rows and in every tile shape."""
    x, w = rand(M, K, seed=M).bfloat16(), rand(N, K, seed=N, scale=K ** -0.5).bfloat16()
    assert ops.gemm_gelu_supported(x.to(DEV), w.to(DEV))
    want = torch.nn.functional.gelu(x.double() @ w.double().t())
    algos = [0] + ([ops.ALGO_TILE + t for t in (64, 128, 256, 512) if t < 256 or M > 128] if M > 64 else [])
    for algo in algos:
        got = ops.gemm(x.to(DEV), w.to(DEV), epilogue=ops.EPI_GELU, algo=algo)
        assert got.dtype == torch.bfloat16
        # (a bfloat16 rounding of the result, and sqrt(K) roundings of 2^-24 of sums of size one to three before it)
        assert ((got.cpu().double() - want).abs() <= want.abs() * 2.0 ** -8 + 2.0 ** -22 * K ** 0.5).all(), algo


@pytest.mark.parametrize("dtype,tol", [(torch.float32, 1e-6), (torch.bfloat16, 2.0 ** -8)])
@pytest.mark.parametrize("W,n", [(4, 1), (20, 8), (256, 5), (260, 6), (1028, 9)])
def test_token_shift_in_whole_pieces(ops, dtype, tol, W, n):
    """Four columns a thread: columns that end inside a block's, one to nine blends (eight fit the registers), portions and
    single rows, states that are not touched."""
    mu = torch.rand(n, W, generator=torch.Generator().manual_seed(W))
    state = torch.full((3, W + 4), 7.0, device=DEV)
    first = rand(3, W, seed=n)
    state[:, :W] = first.to(DEV)
    prev = {s: first[s].double() for s in range(3)}
    for lens, single in (((5, 0, 2), False), ((1, 0, 1), True), ((1, 0, 300), False)):
        seq = sum(([s] * k for s, k in enumerate(lens)), [])
        x = rand(len(seq), W, seed=len(seq)).to(dtype)
        y = ops.token_shift(x.to(DEV), mu.to(DEV), state, torch.tensor(seq, dtype=torch.int32, device=DEV), single_rows=single)
        for t, s in enumerate(seq):
            h = x[t].double()
            want = h + (prev[s] - h) * mu.double()
            assert ((y[:, t].cpu().double() - want).abs() <= tol * (h.abs() + prev[s].abs()) + 1e-30).all(), (lens, t)
            prev[s] = h
    for s in range(3):
        assert torch.equal(state[s, :W].cpu().double(), prev[s])
    assert float(state[:, W:].min()) == 7.0


@pytest.mark.parametrize("dtype,tol", [(torch.float32, 2e-6), (torch.bfloat16, 2.0 ** -8)])
@pytest.mark.parametrize("N,groups", [(4, 1), (2048, 1), (2052, 1), (8192, 1), (8, 2), (96, 3), (2048, 16), (4096, 16), (4100, 1), (4096, 64),
                                      (8192, 32), (2560, 10), (8196, 1)])
def test_gated_norm_in_registers(ops, dtype, tol, N, groups):
    """A row in registers: one group, groups of one to 64 lanes, rows that end inside a thread's pieces, the longest and one more."""
    x, w, gate = rand(3, N, seed=N) * 3, 1 + 0.3 * rand(N, seed=1), rand(3, 2 * N + 8, seed=2).to(dtype)
    off = -N % 8 + N                                       # (whole 16-byte pieces from the row's start)
    gate = gate[:, off:off + N]
    want = rms_of(x.double().view(3, groups, -1)).view(3, N) * w.double() * torch.nn.functional.silu(gate.double()) * 0.5
    got = ops.gated_norm(x.to(DEV), w.to(DEV), 1e-5, groups, dtype, gate=gate.to(DEV), gate_act=ops.GATE_SILU, scale=0.5)
    assert got.dtype == dtype and ((got.cpu().double() - want).abs() <= tol * want.abs() + 1e-7).all()


@pytest.mark.parametrize("hkv,G,dk,dv,dc,window", [(1, 1, 8, 8, 8, -100), (1, 8, 64, 64, 64, 0), (3, 2, 12, 20, 24, -1024), (4, 4, 128, 128, 128, -600),
                                                   (5, 3, 100, 128, 128, 70), (8, 8, 128, 64, 128, -300), (16, 1, 72, 4, 80, 0),
                                                   (16, 2, 64, 64, 64, -200)])
def test_talking_heads_in_registers(ops, hkv, G, dk, dv, dc, window):
    """A tile of keys in registers: one to sixteen key/value heads (four, two or one wave each) of one to eight queries, heads
    that end inside a lane's piece, windows, chunks and neither, tokens with keys in one tile and in several splits.  What
    lies behind a token's keys or beyond a row's numbers is not a number and must not be used."""
    hq, P, L = hkv * G, 16, 700
    q = rand(L, hq, dc, seed=hq).bfloat16()
    k, v = rand(L, hkv, dc, seed=dk).bfloat16(), rand(L, hkv, dc, seed=dv + 1).bfloat16()
    talk, bias = torch.eye(hq) + 0.3 * rand(hq, hq, seed=3) / hq ** 0.5, rand(40, hq, seed=4)
    pages = -(-L // P)
    order = torch.randperm(pages + 3, generator=torch.Generator().manual_seed(5))[:pages]
    cache = torch.full((pages + 3, 2, hkv, P, dc), float("nan"), dtype=torch.bfloat16)
    last = 650
    kk = k.clone()
    kk[:, :, (dk + 3) // 4 * 4:] = float("nan")
    kk[:, :, dk:(dk + 3) // 4 * 4] = 0
    for j in range(last + 1):
        cache[order[j // P], 0, :, j % P] = kk[j]
        cache[order[j // P], 1, :, j % P, :dv] = v[j, :, :dv]
    pos = [0, 1, 15, 63, 64, 65, 199, 200, 299, 511, 599, 600, last]
    kw = dict(window=window) if window >= 0 else dict(chunk=-window)
    got = ops.attention_talk(q[pos].to(DEV), cache.to(DEV), torch.tensor(pos, dtype=torch.int32, device=DEV),
                             torch.zeros(len(pos), dtype=torch.int32, device=DEV), order.int()[None].to(DEV), dk ** -0.5, dk, dv,
                             bias=bias.to(DEV), talk=talk.to(DEV), **kw).cpu().double().view(len(pos), hq, dv)
    for i, p in enumerate(pos):
        lo = max(0, p - window + 1) if window > 0 else (p // -window * -window if window < 0 else 0)
        kd, vd = k[lo:p + 1, :, :dk].double(), v[lo:p + 1, :, :dv].double()
        s = torch.stack([kd[:, h // G] @ q[p, h, :dk].double() for h in range(hq)]) * dk ** -0.5
        s = talk.double() @ (s + bias.double()[(p - torch.arange(lo, p + 1)).clamp(max=39)].t())
        w = torch.softmax(s, -1)
        want = torch.stack([w[h] @ vd[:, h // G] for h in range(hq)])
        # (a bfloat16 rounding of each result; the scores' own errors, some 2^-20, move the weights by as much)
        assert ((got[i] - want).abs() <= want.abs() * 2.0 ** -8 + 2.0 ** -17 * vd.abs().max()).all(), p


@pytest.mark.parametrize("hq,hkv,D,window", [(4, 4, 128, 0), (16, 2, 64, 0), (6, 2, 128, 40), (8, 8, 64, 200), (16, 1, 128, 130)])
@pytest.mark.parametrize("copies", [1, 40])
def test_decode_attention_by_one_wave_and_by_four(ops, hq, hkv, D, window, copies):
    """Single new tokens with a split's tiles dealt to four waves (few tokens) and to one (many), with the step before folded in and
    without: positions at the edges of tiles and splits, a wave without a tile, the token's own key alone in its split."""
    P, pos = 16, [0, 1, 15, 16, 17, 48, 63, 64, 127, 128, 129, 255, 256, 300]
    n = len(pos)
    pages = [p // P + 1 for p in pos]
    order = torch.randperm(sum(pages), generator=torch.Generator().manual_seed(7)).int()
    table, at = torch.full((n, max(pages)), -1, dtype=torch.int32), 0
    cache = torch.full((sum(pages), 2, hkv, P * D), float("nan"), dtype=torch.bfloat16)     # (a key tile [P][D], a value tile [D][P])
    q, ks, vs = rand(n, hq, D, seed=hq).bfloat16(), [], []
    for i, p in enumerate(pos):
        k, v = rand(p + 1, hkv, D, seed=20 + i).bfloat16(), rand(p + 1, hkv, D, seed=60 + i).bfloat16()
        ids = order[at:at + pages[i]]
        at += pages[i]
        table[i, :pages[i]] = ids
        for j in range(p + 1):
            page = cache[ids[j // P]]
            page[0].view(hkv, P, D)[:, j % P] = k[j]
            page[1].view(hkv, D, P)[:, :, j % P] = v[j]
        ks.append(k)
        vs.append(v)
    cache = cache.view(-1, 2, hkv, P, D).to(DEV)
    rows = torch.arange(n).repeat(copies)
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device=DEV)
    positions, seq = i32(pos)[rows.to(DEV)], rows.int().to(DEV)
    scale = 1.5 / D ** 0.5
    out = ops.attention(q[rows].to(DEV), cache, positions, seq, table.to(DEV), scale, window, dec_tokens=i32(range(len(rows))),
                        max_dec_position=max(pos)).cpu()
    qkv = torch.stack([torch.cat([q[i].flatten(), ks[i][-1].flatten(), vs[i][-1].flatten()]) for i in range(n)])
    fused = ops.attention_decode_fused(qkv[rows].to(DEV), hq, cache, positions, seq, table.to(DEV), scale, window, None, max(pos),
                                       None, None, 1e-6, None, None).cpu()
    for i, p in enumerate(pos):
        lo = max(0, p - window + 1) if window else 0
        k, v = ks[i][lo:].double(), vs[i][lo:].double()
        w = torch.softmax(torch.stack([k[:, h * hkv // hq] @ q[i, h].double() for h in range(hq)]) * scale, -1)
        want = torch.stack([w[h] @ v[:, h * hkv // hq] for h in range(hq)])
        # (the weights and the result are rounded to bfloat16: 2^-9 of each weight times its value, and of the result)
        bound = 2.0 ** -8 * (torch.stack([w[h] @ v[:, h * hkv // hq].abs() for h in range(hq)]) + want.abs())
        for got in (out, fused):
            for c in (0, copies - 1):
                assert ((got.view(len(rows), hq, D)[c * n + i].double() - want).abs() <= bound).all(), (p, c)


@pytest.mark.parametrize("hq,hkv,D,page", [(4, 4, 128, 16), (16, 2, 64, 48), (6, 2, 128, 32), (16, 1, 64, 16)])
@pytest.mark.parametrize("window,keep_first,softcap", [(0, 0, 0.0), (70, 0, 0.0), (150, 20, 0.0), (33, 300, 25.0), (0, 0, 30.0)])
def test_decode_attention_of_a_token_alone_and_in_company(ops, hq, hkv, D, page, window, keep_first, softcap):
    """Few tokens' splits are shared by four waves, many tokens' have one each: a token gets the same bits either way, with
    the step before folded in (the new key and value in the cache too) and without.  What lies behind a request's keys or is
    not seen may be anything."""
    pos = [0, 1, 15, 16, 17, 48, 63, 64, 127, 128, 129, 143, 255, 256, 300, 383, 384, 640]
    n, copies, most = len(pos), 30, max(pos)
    pages = [p // page + 1 for p in pos]
    order = torch.randperm(sum(pages), generator=torch.Generator().manual_seed(7)).int()
    table, at = torch.full((n, max(pages)), -1, dtype=torch.int32), 0
    cache = torch.full((sum(pages), 2, hkv, page * D), float("nan"), dtype=torch.bfloat16)
    for i, p in enumerate(pos):
        table[i, :pages[i]] = order[at:at + pages[i]]
        at += pages[i]
        k, v = rand(p + 1, hkv, D, seed=20 + i, scale=2.0).bfloat16(), rand(p + 1, hkv, D, seed=60 + i).bfloat16()
        for j in range(p + 1):
            here = cache[table[i, j // page]]
            here[0].view(hkv, page, D)[:, j % page] = k[j]
            here[1].view(hkv, D, page)[:, :, j % page] = v[j]
    cache, table = cache.view(-1, 2, hkv, page, D).to(DEV), table.to(DEV)
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device=DEV)
    rows = list(range(n)) * copies
    positions = i32([pos[i] for i in rows])
    q = rand(n, hq, D, seed=hq).bfloat16()[rows].to(DEV)
    seen = dict(window=window, keep_first=keep_first, softcap=softcap, max_dec_position=most)
    every = ops.attention(q, cache, positions, i32(rows), table, 0.15, dec_tokens=i32(range(len(rows))), **seen)
    assert len(rows) * hkv * (most // 128 + 1) > 512 >= hkv * (most // 128 + 1)
    for i in range(n):
        alone = ops.attention(q, cache, positions, i32(rows), table, 0.15, dec_tokens=i32([i]), **seen)
        assert torch.equal(alone[i], every[i]) and torch.equal(every[i], every[i + n]), pos[i]
    if keep_first or softcap:
        return
    qkv = rand(n, (hq + 2 * hkv) * D, seed=8).bfloat16()[rows].to(DEV)
    qw, kw, turn = 1 + rand(D, seed=1).to(DEV) / 4, 1 + rand(D, seed=2).to(DEV) / 4, torch.rand(most + 1, D, device=DEV)
    slots = [-1 if i == 3 else int(table[i, p // page]) * page + p % page for i, p in enumerate(pos)]
    fused = lambda c, which: ops.attention_decode_fused(qkv, hq, c, positions, i32(rows), table, 0.15, window, i32(which), most, qw, kw, 1e-6,
                                                        turn, i32(slots + [-1] * (len(rows) - n)))
    together = cache.clone()
    every = fused(together, range(len(rows)))
    one_by_one = cache.clone()
    for i in range(n):
        assert torch.equal(fused(one_by_one, [i])[i], every[i]), pos[i]
    assert torch.equal(torch.nan_to_num(one_by_one.float()), torch.nan_to_num(together.float()))
    assert not torch.isnan(every).any()


@pytest.mark.parametrize("E,K,F", [(16, 264, 192), (6, 2048, 544), (40, 512, 96)])
@pytest.mark.parametrize("T", [2, 9, 48])
def test_experts_of_few_rows_in_steps_of_k(ops, E, K, F, T):
    """The experts' products with eight steps of K in flight (few blocks) and with four: against the 64-bit products, and a token the
    same bits alone and in company."""
    top = 2
    x, wg, wd = rand(T, K, seed=1).bfloat16(), rand(E, 2 * F, K, seed=2, scale=K ** -0.5).bfloat16(), rand(E, K, F, seed=3, scale=F ** -0.5).bfloat16()
    ids = torch.stack([torch.randperm(E, generator=torch.Generator().manual_seed(t))[:top] for t in range(T)]).int()
    weights = torch.rand(T, top, generator=torch.Generator().manual_seed(9)) + 0.1
    run = lambda n: ops.moe_experts(x[:n].to(DEV), ids[:n].to(DEV), weights[:n].to(DEV), wg.to(DEV), wd.to(DEV)).cpu()
    got, alone = run(T), run(1)
    assert got.shape == (top, T, K) and torch.equal(alone[:, 0], got[:, 0])
    for t in range(T):
        for j in range(top):
            gate, up = (wg[ids[t, j]].double() @ x[t].double()).split(F)
            mid = torch.nn.functional.silu(gate) * up
            down = wd[ids[t, j]].double()
            want = weights[t, j].double() * (down @ mid)
            # (the middle rounded to bfloat16, 2^-9 of each; the 32-bit sums far below)
            bound = weights[t, j].double() * (2.0 ** -8 * (down.abs() @ mid.abs()) + 1e-4)
            assert ((got[j, t].double() - want).abs() <= bound).all(), (t, j)


@pytest.mark.parametrize("T,H,N,K", [(1, 16, 128, 512), (1, 3, 20, 8), (2, 2, 64, 40), (17, 5, 130, 256), (32, 1, 16, 264), (33, 2, 128, 520), (70, 3, 40, 72)])
def test_products_of_heads_in_steps_of_k(ops, T, H, N, K):
    """Eight steps of K asked for together (few rows) and two (many): sums of whole numbers far below 2^24, rounded once."""
    g = torch.Generator().manual_seed(K)
    x, w = torch.randint(-3, 4, (T, H, K), generator=g).bfloat16(), torch.randint(-3, 4, (H, N, K), generator=g).bfloat16()
    out = torch.empty(T, H, N, dtype=torch.bfloat16, device=DEV)
    ops.gemm_heads(x.to(DEV), w.to(DEV), out)
    want = torch.stack([x[:, h].float() @ w[h].float().t() for h in range(H)], 1).bfloat16()
    assert torch.equal(out.cpu(), want)


@pytest.mark.parametrize("H,R,dr", [(16, 512, 64), (5, 8, 8), (16, 64, 64), (3, 120, 72), (16, 256, 64), (16, 200, 48), (17, 128, 64), (48, 64, 32)])
@pytest.mark.parametrize("window", [0, 50])
def test_latent_attention_of_single_tokens(ops, H, R, dr, window):
    """Four waves share a token's heads (up to 16 of them) or take a group each: latents of every size class, one key, tiles' edges,
    many splits and splits without keys."""
    before = [0, 30, 31, 32, 200, 1100]
    cache, table, pos, seq, own = latent_rows(before, [1] * len(before), R, dr, 16, 50)
    q = rand(len(before), H, R + dr, seed=9).bfloat16()
    scale = (R + dr) ** -0.5
    for rows in (list(range(len(before))), [5], list(range(len(before))) * 12):
        got = ops.latent_attention(q[rows].to(DEV), cache, pos[rows], seq[rows], table, R, scale, window=window).cpu().double()
        for j, i in enumerate(rows[:len(before)]):
            c = own[i][max(0, len(own[i]) - window) if window else 0:]
            w = torch.softmax(q[i].double() @ c.t() * scale, -1)
            want = w @ c[:, :R]
            assert ((got[j] - want).abs() <= 2.0 ** -8 * (w @ c[:, :R].abs() + want.abs())).all(), (i, rows[:2])


@pytest.mark.parametrize("H,R,dr", [(32, 512, 64), (48, 256, 64), (16, 512, 64)])
@pytest.mark.parametrize("window", [0, 700])
def test_latent_splits_are_merged_in_one_order(ops, H, R, dr, window):
    """Up to eight single tokens have as many splits each as one; the merge by four parts a thread group (few heads) and by one thread
    (many) adds them up in the same order: a token gets the same bits alone and with seven others."""
    before = [0, 30, 200, 640, 900, 1100, 1500, 77]
    cache, table, pos, seq, own = latent_rows(before, [1] * len(before), R, dr, 16, 50)
    q = rand(len(before), H, R + dr, seed=9).bfloat16().to(DEV)
    scale = (R + dr) ** -0.5
    every = ops.latent_attention(q, cache, pos, seq, table, R, scale, window=window)
    for i in range(len(before)):
        assert torch.equal(ops.latent_attention(q[i:i + 1], cache, pos[i:i + 1], seq[i:i + 1], table, R, scale, window=window)[0], every[i]), i


@pytest.mark.parametrize("tile", [64, 128, 256, 512])
@pytest.mark.parametrize("page", [16, 64])
def test_qkv_product_stores_values_behind_other_rows(ops, tile, page):
    """Values go to the cache in pieces of eight tokens wherever eight slots lie side by side from a multiple of eight on: rows whose
    slots are scattered, absent, in runs that begin in the middle of a piece and of a tile, whole pages and runs in descending
    order.  Sums of whole numbers, rounded once; what is not named stays as it was."""
    hq, hkv, K, M = 2, 3, 64, 410
    slots = [5, 900, 17, -1, 40] + list(range(61, 150)) + [-1] * 3 + list(range(200, 233)) + list(range(448, 256, -1)) + list(range(512, 600))
    assert len(slots) == M
    g = torch.Generator().manual_seed(page)
    x = torch.randint(-3, 4, (M, K), generator=g).bfloat16()
    w = torch.randint(-3, 4, ((hq + 2 * hkv) * 128, K), generator=g).bfloat16()
    cache = torch.full((1024 // page, 2, hkv, page * 128), -0.5, dtype=torch.bfloat16)
    want, y = cache.clone(), (x.float() @ w.float().t()).bfloat16()
    for m, s in enumerate(slots):
        if s >= 0:
            want[s // page, 0].view(hkv, page, 128)[:, s % page] = y[m, hq * 128:(hq + hkv) * 128].view(hkv, 128)
            want[s // page, 1].view(hkv, 128, page)[:, :, s % page] = y[m, (hq + hkv) * 128:].view(hkv, 128)
    got = cache.view(-1, 2, hkv, page, 128).to(DEV)
    q = ops.gemm_qkv(x.to(DEV), w.to(DEV), None, hq, got, torch.zeros(M, dtype=torch.int32, device=DEV), None, None, 1e-6, None,
                     torch.tensor(slots, dtype=torch.int32, device=DEV), tile=tile)
    assert torch.equal(q.cpu().view(M, -1), y[:, :hq * 128])
    assert torch.equal(got.cpu().view(want.shape), want)


@pytest.mark.parametrize("M,N", [(656, 24576), (1601, 10368), (2048, 10240)])
def test_products_in_two_launches(ops, M, N):
    """Products whose last turn of tiles is thin go in two launches over the columns: gate and up with silu, the product itself with a
    bias, and q|k|v (with the cut among the queries and among the values), against the same in one launch of one shape.  Whole
    numbers where nothing is computed on the sums."""
    g = torch.Generator().manual_seed(N)
    K = 2048
    first = ops.gemm_first_columns(M, N, K)
    assert 0 < first < N and first % 256 == 0
    x = torch.randint(-2, 3, (M, K), generator=g).bfloat16().to(DEV)
    w = torch.randint(-2, 3, (N, K), generator=g).bfloat16().to(DEV)
    bias = torch.randint(-9, 9, (N,), generator=g).float().to(DEV)
    want = x.float() @ w.float().t()
    assert torch.equal(ops.gemm(x, w, bias, out_dtype=torch.float32), want + bias)
    gate_up = (x.double() @ w.double().t()).view(M, N // 64, 2, 32) * 2.0 ** -6
    small = (w.float() * 2.0 ** -6).bfloat16()
    act = (torch.nn.functional.silu(gate_up[:, :, 0]) * gate_up[:, :, 1]).reshape(M, N // 2)
    got = ops.gemm(x, small, epilogue=ops.EPI_SILU_MUL_IL).double()
    assert ((got - act).abs() <= act.abs() * 2.0 ** -8 + 2.0 ** -20).all()
    heads, at = N // 128, torch.arange(M, dtype=torch.int32, device=DEV)
    most = max(d for d in range(1, heads // 3 + 1) if heads % d == 0)
    assert (heads - most) * 128 < first < N - 256                        # (among the values of most heads, among the queries of one)
    for hkv in (1, most):
        hq = heads - 2 * hkv
        cache = [torch.zeros(M // 16 + 1, 2, hkv, 16, 128, dtype=torch.bfloat16, device=DEV) for _ in range(2)]
        q = [ops.gemm_qkv(x, w, None, hq, c, at, None, None, 1e-6, None, at, tile=t) for c, t in zip(cache, (0, 128))]
        assert torch.equal(q[0], q[1]) and torch.equal(cache[0], cache[1])
        assert torch.equal(q[0].view(M, -1).float(), want[:, :hq * 128].bfloat16().float())


@pytest.mark.parametrize("M,N", [(1600, 5120), (1601, 5176)])
def test_gelu_products_in_two_launches(ops, M, N):
    """The gelu's product where its last turn of tiles is thin, against one launch of one shape and 64 bits."""
    K = 2048
    first = ops.gemm_first_columns(M, N, K, gelu=True)
    assert 0 < first < N and first % 256 == 0
    x, w = rand(M, K, seed=M).bfloat16().to(DEV), rand(N, K, seed=N, scale=K ** -0.5).bfloat16().to(DEV)
    got = ops.gemm(x, w, epilogue=ops.EPI_GELU)
    assert torch.equal(got, ops.gemm(x, w, epilogue=ops.EPI_GELU, algo=ops.ALGO_TILE + 128))
    want = torch.nn.functional.gelu(x.double() @ w.double().t())
    # (a bfloat16 rounding of the result, and sqrt(K) roundings of 2^-24 of sums of size one to three before it)
    assert ((got.double() - want).abs() <= want.abs() * 2.0 ** -8 + 2.0 ** -22 * K ** 0.5).all()


@pytest.mark.parametrize("hq,hkv,D,window", [(4, 2, 128, 0), (3, 1, 16, 0), (6, 2, 48, 100), (2, 2, 256, 0), (20, 1, 64, 37), (4, 4, 144, 0)])
def test_float32_attention_in_eight_walks(ops, hq, hkv, D, window):
    """Few tokens (eight waves, a walk each) and many (four waves, two walks each): against 64 bits, and the same bits."""
    P, L = 16, 430
    k, v, q = rand(L, hkv, D, seed=1), rand(L, hkv, D, seed=2), rand(L, hq, D, seed=3)
    pages = -(-L // P)
    order = torch.randperm(pages + 2, generator=torch.Generator().manual_seed(4))[:pages].int()
    cache = torch.full((pages + 2, 2, hkv, P * D), float("nan"))
    for j in range(L):
        page = cache[order[j // P]]
        page[0].view(hkv, P, D)[:, j % P] = k[j]
        page[1].view(hkv, D, P)[:, :, j % P] = v[j]
    cache, table = cache.view(-1, 2, hkv, P, D).to(DEV), order[None].to(DEV)
    scale = D ** -0.5

    def run(rows):
        r = torch.tensor(rows, dtype=torch.int32, device=DEV)
        return ops.attention(q[rows].to(DEV), cache, r, torch.zeros_like(r), table, scale, window).cpu()

    every = run(list(range(L)))
    for p in (0, 1, 15, 16, 63, 64, 127, 128, 200, 255, 429):
        got = run([p])[0]
        lo = max(0, p - window + 1) if window else 0
        w = torch.softmax(torch.stack([k[lo:p + 1, h * hkv // hq].double() @ q[p, h].double() for h in range(hq)]) * scale, -1)
        want = torch.stack([w[h] @ v[lo:p + 1, h * hkv // hq].double() for h in range(hq)])
        size = torch.stack([w[h] @ v[lo:p + 1, h * hkv // hq].double().abs() for h in range(hq)])
        # (scores of a few units and the sums: some sqrt(keys + D) roundings of 2^-24 each)
        assert ((got.double() - want).abs() <= 2.0 ** -24 * 4 * (p + 1 + D) ** 0.5 * size + 1e-30).all(), p
        assert torch.equal(got, every[p]), p


@pytest.mark.parametrize("taps", [2, 3, 4, 8])
@pytest.mark.parametrize("H", [4, 260, 1028, 157292])
def test_short_convolution_by_eight_rows(ops, taps, H):
    """Four channels of eight rows a thread (the most channels) and a thread a number: portions that begin and end anywhere in a block's rows, shorter than the taps and longer
    than blocks, continued from step to step; what no row names stays as it was."""
    w = rand(H, taps, seed=taps)
    state = torch.full((5, taps - 1, H), 7.0, device=DEV)
    state[:4] = 0
    past = {s: torch.zeros(0, H) for s in range(4)}
    for step, lens in enumerate(([5, 0, 1, 12], [1, 3, 0, 8], [9, 2, 30, 1], [2, 1, 1, 1])):
        rows = {s: rand(n, H, seed=10 * step + s) for s, n in enumerate(lens) if n}
        seq = torch.tensor(sum(([s] * lens[s] for s in rows), []), dtype=torch.int32, device=DEV)
        got = ops.short_conv(torch.cat(list(rows.values())).to(DEV), w.to(DEV), state, seq, torch.float32).cpu()
        want, size = [], []
        for s, x in rows.items():
            full = torch.cat([torch.zeros(taps - 1, H), past[s], x]).double()
            past[s] = torch.cat([past[s], x])
            n0 = len(full) - len(x)
            for to, f, wd in ((want, full, w.double()), (size, full.abs(), w.double().abs())):
                to.append(torch.stack([f[n0 + i] + sum(wd[:, taps - 1 - k] * f[n0 + i - k] for k in range(taps)) for i in range(len(x))]))
            last = torch.cat([torch.zeros(taps - 1, H), past[s]])[-(taps - 1):]
            assert torch.equal(state[s].cpu(), last), (step, s)
        # (a multiply-add a tap, each rounded by 2^-24 of a partial sum, which is at most the sum of the sizes of its terms)
        assert ((got.double() - torch.cat(want)).abs() <= 2.0 ** -24 * taps * torch.cat(size)).all(), step
    assert float(state[4].min()) == 7.0


@pytest.mark.parametrize("taps", [2, 4, 8])
@pytest.mark.parametrize("H,lens", [(260, (1500, 0, 8, 1700)), (1028, (5, 401, 1, 377)), (157292, (2, 0, 1, 2))])
def test_short_convolution_of_many_rows_as_of_few(ops, taps, H, lens):
    """Steps with rows and channels enough for eight rows a thread, and the same rows a few at a time (a thread a number): the same
    bits, in the results and in the state, over three steps of portions that end anywhere."""
    w = rand(H, taps, seed=taps).to(DEV)
    many = torch.zeros(5, taps - 1, H, device=DEV)
    few = many.clone()
    for step in range(3):
        n = [max(0, k - step * (k > 4)) for k in lens]
        assert sum(n) * H >= 3 << 18
        x = torch.randn(sum(n), H, device=DEV, generator=torch.Generator(DEV).manual_seed(step))
        seq = torch.repeat_interleave(torch.arange(4), torch.tensor(n)).int().to(DEV)
        got = ops.short_conv(x, w, many, seq, torch.float32)
        piece = max(1, (3 << 18) // H - 1)
        parts = [ops.short_conv(x[a:a + piece], w, few, seq[a:a + piece], torch.float32) for a in range(0, len(x), piece)]
        assert torch.equal(got, torch.cat(parts)) and torch.equal(many, few), step


@pytest.mark.parametrize("hq,hkv,D", [(16, 4, 128), (30, 6, 72), (24, 8, 96)])
def test_whole_norms_in_one_order(ops, hq, hkv, D):
    """The norm over a whole projection by 1024 threads (few rows) and by 256 (many): a row gets the same bits."""
    T = 700
    y = rand(T, (hq + 2 * hkv) * D, seed=D).bfloat16().to(DEV)
    wq, wk = 1 + rand(hq * D, seed=1).to(DEV) / 4, 1 + rand(hkv * D, seed=2).to(DEV) / 4
    at = torch.arange(T, dtype=torch.int32, device=DEV)

    def run(rows):
        cache = torch.zeros(T // 16 + 1, 2, hkv, 16, D, dtype=torch.bfloat16, device=DEV)
        q = ops.qkv_norm_store(y[rows], hq, hkv, D, D, cache, at[rows], qk_norm=ops.QK_NORM_WHOLE, q_weight=wq, k_weight=wk, qk_eps=1e-5)
        return q, cache

    q, cache = run(slice(0, T))
    some = slice(130, 140)
    q_some, cache_some = run(some)
    assert torch.equal(q_some, q[some])
    here = cache_some.abs().sum((0, 1, 2, 4)) > 0
    assert here.any()
    for t in range(130, 140):
        assert torch.equal(cache_some[t // 16, :, :, :, :][0][:, t % 16], cache[t // 16][0][:, t % 16]), t


@pytest.mark.parametrize("D,T", [(128, 200), (128, 700), (64, 200), (64, 300)])
def test_talking_heads_of_one_key_value_head(ops, D, T):
    """Eight queries on one key/value head: many rows go several a block, few a block each; both against 64 bits."""
    hq, P = 8, 16
    q, k, v = rand(T, hq, D, seed=1).bfloat16().to(DEV), rand(T, D, seed=2).bfloat16().to(DEV), rand(T, D, seed=3).bfloat16().to(DEV)
    talk, bias = (torch.eye(hq) + 0.1 * rand(hq, hq, seed=4)).to(DEV), rand(40, hq, seed=5).to(DEV)
    cache = torch.full((T // P + 1, 2, 1, P, D), float("nan"), dtype=torch.bfloat16, device=DEV)
    cache[torch.arange(T) // P, 0, 0, torch.arange(T) % P] = k
    cache[torch.arange(T) // P, 1, 0, torch.arange(T) % P] = v
    pos = torch.arange(T, dtype=torch.int32, device=DEV)
    seq, table = torch.zeros_like(pos), torch.arange(T // P + 1, dtype=torch.int32, device=DEV)[None]
    kw = dict(chunk=1024, bias=bias, talk=talk)
    every = ops.attention_talk(q, cache, pos, seq, table, D ** -0.5, D, D, **kw)
    few = torch.zeros_like(every)
    some = pos[T - 20:].contiguous()
    ops.attention_talk(q, cache, pos, seq, table, D ** -0.5, D, D, out=few, tokens=some, **kw)
    d = (pos[:, None] - pos[None]).long()
    s = (q.double().transpose(0, 1) @ k.double().t()) * D ** -0.5 + bias.double()[d.clamp(0, 39)].permute(2, 0, 1)
    s = (talk.double() @ s.reshape(hq, -1)).view(hq, T, T).masked_fill(d < 0, float("-inf"))
    w = torch.softmax(s, -1)
    want = (w @ v.double()).transpose(0, 1).reshape(T, -1)
    # (a bfloat16 rounding of each result; the scores' own errors, some 2^-20, move the weights by as much)
    bound = want.abs() * 2.0 ** -8 + 2.0 ** -17 * v.double().abs().max()
    assert ((every.double() - want).abs() <= bound).all()
    assert ((few.double() - want).abs() <= bound)[T - 20:].all()


def test_prefill_attention_takes_two_groups_where_one_walk_decides(ops):
    """Blocks once to twice the compute units: two wave groups for one prompt from its start or beside short ones, one for walks of
    one length, whether short or deep in a context, for windows and where the keys are not known; two for few blocks."""
    units = torch.cuda.get_device_properties(0).multi_processor_count
    rows = ops.prefill_tile_rows(32, 8)
    tiles = lambda n: -(-n // (4 * rows)) * 4
    blocks = lambda n: tiles(n) // 4 * 8 * (4 // (32 // rows))
    assert units < blocks(2048) <= 2 * units and blocks(1000) <= units < 2 * units < blocks(3000)
    groups = lambda n, keys, window=0: ops.prefill_groups_of(tiles(n), 32, 8, window, keys)
    assert groups(2048, 2048) == 2 and groups(2048, 1600) == 2
    assert groups(2048, 128) == groups(2048, 512) == groups(2048, 8192) == groups(2048, 0) == groups(2048, 2048, 512) == 1
    assert groups(1000, 100) == groups(1000, 30000) == 2 and groups(3000, 3000) == 1


def test_parts_of_a_product_stay_within_their_bytes(ops):
    """However many rows a step has, the partial products that are asked for take 512 MiB at the most."""
    for n, k in ((5120, 25600), (4096, 12288), (5120, 8192), (1024, 3072)):
        w = torch.empty(n, k, dtype=torch.bfloat16, device=DEV)
        for rows in (1, 64, 512, 2048, 8192, 12288, 16384, 32768, 65536):
            splits = ops.gemm_branch_splits_for(rows, w, torch.bfloat16)
            assert splits * rows * n * 4 <= 512 << 20, (rows, n, k, splits)


@pytest.mark.parametrize("K", [64, 72, 128, 200, 320, 1096])
def test_tiled_products_at_the_ends_of_their_stages(ops, K):
    """One stage of 64 of K and several, odd and even numbers, whole and not, in every tile shape, rows and columns just beyond and
    short of a tile, and two cuts of K; NaN and infinities beside the operands change nothing."""
    for M, N in ((65, 136), (129, 120), (257, 264), (255, 256)):
        xs, ws = (torch.full((r + 2, K), float("nan"), dtype=torch.bfloat16) for r in (M, N))
        xs[0], ws[0] = float("inf"), float("-inf")
        xs[1:-1], ws[1:-1] = rand(M, K, seed=M + K, dtype=torch.bfloat16), rand(N, K, seed=N + K, dtype=torch.bfloat16)
        x, w = xs.to(DEV)[1:-1], ws.to(DEV)[1:-1]
        want = xs[1:-1].double() @ ws[1:-1].double().t()
        # (K products summed in 32-bit: some sqrt(K) units of 2^-24 of the sum of their sizes; 2^-20 bounds it)
        bound = 2.0 ** -20 * (xs[1:-1].double().abs() @ ws[1:-1].double().abs().t())
        for rows in (64, 65, 128, 256, 512):
            got = ops.gemm(x, w, out_dtype=torch.float32, algo=ops.ALGO_TILE + rows)
            assert ((got.cpu().double() - want).abs() <= bound).all(), (M, N, K, rows)
            if K > 64:
                parts = ops.gemm(x, w, epilogue=ops.EPI_PARTIAL, splits=2, algo=ops.ALGO_TILE + rows)
                assert ((parts.cpu().double().sum(0) - want).abs() <= bound).all(), (M, N, K, rows)


def odd(t):
    """The same numbers in a tensor that begins at an odd element."""
    t = torch.cat([t.new_zeros(1), t.reshape(-1)])[1:].view(t.shape)
    assert t.data_ptr() % 4 == 2
    return t


@pytest.mark.parametrize("M,N,K", [(200, 192, 328), (65, 64, 64), (255, 320, 72), (300, 256, 1160)])
def test_tiled_products_of_operands_at_any_address(ops, M, N, K):
    """Operands that begin at an odd element: the bits of aligned ones, in every tile shape, as a plain product, gate and up, gelu and in
    cuts of K."""
    x, w = rand(M, K, seed=1, dtype=torch.bfloat16).to(DEV), rand(N, K, seed=2, dtype=torch.bfloat16).to(DEV)
    bias = rand(N, seed=3).to(DEV)
    forms = [dict(), dict(out_dtype=torch.float32, bias=bias), dict(epilogue=ops.EPI_SILU_MUL_IL), dict(epilogue=ops.EPI_SILU_MUL_IL, bias=bias),
             dict(epilogue=ops.EPI_GELU)] + ([dict(epilogue=ops.EPI_PARTIAL, splits=2)] if K > 64 else [])
    for rows in (0, 64, 65, 128, 256, 512):
        for form in forms:
            run = lambda a, b: ops.gemm(a, b, algo=ops.ALGO_TILE + rows if rows else ops.ALGO_AUTO, **form)
            want = run(x, w)
            for a, b in ((odd(x), w), (x, odd(w)), (odd(x), odd(w))):
                assert torch.equal(run(a, b), want), (rows, form)


@pytest.mark.parametrize("M", [17, 40, 64])
def test_few_rows_of_operands_at_any_address_against_a_large_matrix(ops, M):
    """17 to 64 rows by the tiles: plain, gate and up (a matrix of few tile columns: a longer ring), in cuts of K."""
    N, K = 4096, 4160
    x, w = rand(M, K, seed=M, dtype=torch.bfloat16).to(DEV), rand(N, K, seed=2, dtype=torch.bfloat16).to(DEV)
    assert ops.gemm_partial_preferred(x, w)
    for form in (dict(), dict(epilogue=ops.EPI_SILU_MUL_IL), dict(epilogue=ops.EPI_PARTIAL, splits=5)):
        assert torch.equal(ops.gemm(odd(x), odd(w), **form), ops.gemm(x, w, **form)), form


@pytest.mark.parametrize("tile", [0, 64, 128, 256, 512])
def test_query_key_value_products_of_operands_at_any_address(ops, tile):
    M, K, hq, hkv, P = 150, 200, 4, 2, 16
    x, w = rand(M, K, seed=1, dtype=torch.bfloat16).to(DEV), rand((hq + 2 * hkv) * 128, K, seed=2, dtype=torch.bfloat16).to(DEV)
    norms = (1 + 0.1 * rand(2, 128, seed=3)).to(DEV)
    table, pos = rand(M, 128, seed=4).to(DEV), torch.arange(M, dtype=torch.int32, device=DEV)
    got = []
    for a, b in ((x, w), (odd(x), odd(w))):
        cache = torch.zeros(M // P + 1, 2, hkv, P, 128, dtype=torch.bfloat16, device=DEV)
        got.append((ops.gemm_qkv(a, b, None, hq, cache, pos, norms[0].contiguous(), norms[1].contiguous(), 1e-6, table, pos, tile=tile), cache))
    assert torch.equal(got[0][0], got[1][0]) and torch.equal(got[0][1], got[1][1]) and got[0][1].any()


@pytest.mark.parametrize("act", ["gated", "relu_sq"])
def test_grouped_products_of_weights_at_any_address(ops, act):
    """Enough pairs for the grouped rows' tiles."""
    T, E, F, K, top = 300, 8, 96, 136, 4
    x = rand(T, K, seed=1, dtype=torch.bfloat16).to(DEV)
    w_in, w_out = rand(E, (2 if act == "gated" else 1) * F, K, seed=2, dtype=torch.bfloat16).to(DEV), rand(E, K, F, seed=3, dtype=torch.bfloat16).to(DEV)
    ids = torch.stack([torch.randperm(E, generator=torch.Generator().manual_seed(t))[:top] for t in range(T)]).int().to(DEV)
    weights = torch.rand(T, top, generator=torch.Generator().manual_seed(5)).to(DEV)
    for rows in (torch.float32, torch.bfloat16):
        got = [ops.moe_experts(x, ids, weights, a, b, act=act, interleaved=act == "gated", rows_dtype=rows) for a, b in
               ((w_in, w_out), (odd(w_in), odd(w_out)))]
        assert torch.equal(*got) and got[0].any()


@pytest.mark.parametrize("K", [1016, 1024, 2048, 4096, 4160, 12288])
def test_products_whose_parts_are_rounded_are_large(ops, K):
    """A branch's product is handed on in 16 bits only where its rows are many (or K is short); else in 32-bit parts."""
    for N in (1024, 2048, 4096, 5120):
        w = torch.empty(N, K, dtype=torch.bfloat16, device=DEV)
        for M in (65, 300, 512, 1000, 2048, 8192):
            splits = ops.gemm_branch_splits_for(M, w, torch.bfloat16)
            tiles = -(-M // 128) * -(-N // 128)
            assert (splits == 0) == (K < 1024) or (splits == 0 and tiles > 256), (M, N, K, splits)


@pytest.mark.parametrize("M,N,K", [(3300, 5120, 8192), (4600, 4096, 12288), (8192, 5120, 8192)])
def test_products_that_go_in_two_launches_are_not_cut(ops, M, N, K):
    """A branch's product whose last turn of tiles gets a launch of its own is quicker as one 32-bit part than in cuts of K; the same
    bits as in one launch."""
    x, w = rand(M, K, seed=1, dtype=torch.bfloat16).to(DEV), rand(N, K, seed=2, dtype=torch.bfloat16).to(DEV)
    assert ops.gemm_first_columns(M, N, K) > 0 and ops.gemm_branch_splits(x, w) == 1
    parts = ops.gemm(x, w, epilogue=ops.EPI_PARTIAL, splits=1)
    assert torch.equal(parts, ops.gemm(x, w, epilogue=ops.EPI_PARTIAL, splits=1, algo=ops.ALGO_TILE + 128))


@pytest.mark.parametrize("D,P", [(128, 16), (128, 64), (64, 16), (64, 32)])
@pytest.mark.parametrize("groups", [1, 2])
def test_prefill_attention_over_few_and_many_tiles(ops, D, P, groups):
    """Prompts that end inside, at and behind tiles of 32 keys, with fewer tiles than shared memory takes and with more, alone and
    behind keys of an earlier step, with and without a window; what the pages hold beside the keys is NaN."""
    from qwen_engine_amd.parts.attention import prefill_tiles
    hq, hkv = 4, 2
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device=DEV)
    for n, before, window in ((1, 0, 0), (15, 0, 0), (33, 0, 0), (64, 0, 0), (90, 0, 0), (97, 31, 0), (128, 0, 0), (129, 16, 0), (160, 0, 40),
                              (161, 100, 33), (290, 7, 0), (300, 0, 128)):
        L = before + n
        k, v, q = (rand(L, h, D, seed=s + L, dtype=torch.bfloat16) for s, h in ((1, hkv), (2, hkv), (3, hq)))
        pages = -(-L // P)
        cache = torch.full((pages + 1, 2, hkv, P, D), float("nan"), dtype=torch.bfloat16)
        order = torch.randperm(pages, generator=torch.Generator().manual_seed(L)) + 1
        vt = cache[:, 1].view(-1, hkv, D, P)
        for t in range(L):
            cache[order[t // P], 0, :, t % P] = k[t]
            vt[order[t // P], :, :, t % P] = v[t]
        tiles = i32(prefill_tiles([(0, n)], ops.prefill_tile_rows(hq, hkv))).view(-1, 2)
        got = ops.attention(q[before:].contiguous().to(DEV), cache.to(DEV), i32(list(range(before, L))), i32([0] * n), order.int()[None].to(DEV), D ** -0.5, window=window,
                            other_tokens=i32(list(range(n))), other_tiles=tiles, prefill_groups=groups).view(n, hq, D).cpu().double()
        pos, key = torch.arange(before, L)[:, None], torch.arange(L)[None]
        hidden = (key > pos) | ((key <= pos - window) if window else torch.zeros_like(key, dtype=torch.bool))
        for h in range(hq):
            s = (q[before:, h].double() @ k[:, h // 2].double().t() * D ** -0.5).masked_fill(hidden, float("-inf"))
            w = torch.softmax(s, -1)
            want, size = w @ v[:, h // 2].double(), w @ v[:, h // 2].double().abs()
            # (each weight and the result rounded to 8 bits of mantissa: 2^-8 of the sum of the sizes, 2^-8 of the result)
            assert ((got[:, h] - want).abs() <= 2.0 ** -8 * (size + want.abs()) + 1e-6).all(), (n, before, window, h)


@pytest.mark.parametrize("N,K", [(16384, 544), (30001, 544), (16384, 608), (16386, 672), (16390, 992), (20001, 1024)])
def test_float32_logits_sum_in_the_same_order(ops, N, K):
    """Few rows against a matrix of very many (its last block of 16 outputs whole and not, K whole quarters and not): the bits
    that the tiles give a row among many, and those of operands at an odd address."""
    x, w, bias = rand(20, K, seed=K).to(DEV), rand(N, K, seed=N).to(DEV), rand(N, seed=3).to(DEV)
    every = ops.gemm(x, w, bias)
    want = x.cpu().double() @ w.cpu().double().t() + bias.cpu().double()
    bound = 2.0 ** -24 * K ** 0.5 * 4 * (x.cpu().double().abs() @ w.cpu().double().abs().t() + bias.cpu().double().abs())
    for M in (1, 3, 16):
        got = ops.gemm(x[:M].contiguous(), w, bias)
        assert torch.equal(got, every[:M]), M
        assert ((got.cpu().double() - want[:M]).abs() <= bound[:M]).all(), M
    odd = torch.cat([w.new_zeros(1), w.reshape(-1)])[1:].view(N, K)
    assert odd.data_ptr() % 16 == 4 and torch.equal(ops.gemm(x[:2].contiguous(), odd, bias), every[:2])


@pytest.mark.parametrize("D,softcap", [(128, 0.0), (64, 0.0), (128, 20.0), (64, 20.0)])
@pytest.mark.parametrize("offset", [1, 4])
def test_prefill_attention_of_a_cache_at_any_address(ops, D, softcap, offset):
    """A cache that begins at no whole 16-byte piece: the bits of an aligned one, by one wave group a block and by two, with keys in
    segments, with a window, with fewer tiles than shared memory takes and with more."""
    from qwen_engine_amd.parts.attention import prefill_tiles
    hq, hkv, P = 8, 2, 16
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device=DEV)
    for n, before, window, segment in ((5, 0, 0, 0), (97, 31, 0, 0), (161, 100, 33, 0), (290, 7, 0, 0), (70, 1100, 0, 512)):
        L = before + n
        pages = -(-L // P)
        cache = rand(pages, 2, hkv, P, D, seed=L, dtype=torch.bfloat16).to(DEV)
        moved = torch.cat([cache.new_zeros(offset), cache.reshape(-1)])[offset:].view(cache.shape)
        assert moved.is_contiguous() and moved.data_ptr() % 16 == 2 * offset
        q = rand(n, hq, D, seed=L + 1, dtype=torch.bfloat16).to(DEV)
        tiles = i32(prefill_tiles([(0, n)], ops.prefill_tile_rows(hq, hkv))).view(-1, 2)
        order = torch.randperm(pages, generator=torch.Generator().manual_seed(L)).int()[None].to(DEV)
        for groups in (1, 2):
            got = [ops.attention(q, c, i32(list(range(before, L))), i32([0] * n), order, D ** -0.5, window=window, softcap=softcap,
                                 other_tokens=i32(list(range(n))), other_tiles=tiles, prefill_groups=groups,
                                 max_other_keys=L if segment else 0, prefill_segment_keys=segment) for c in (cache, moved)]
            assert torch.isfinite(got[0].float()).all() and torch.equal(got[0], got[1]), (n, before, window, segment, groups)
