"""32-bit products of few rows with the residual sum and the norm in front, or silu(gate) * up behind: the numbers that the kernels one by
one give, bit for bit, and those of 64 bits."""
import pytest
import torch

import qwen_engine_amd  # noqa: F401

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ops():
    from qwen_engine_amd.kernels import ops
    return ops


# (rows of two passes of the norm, groups of one to four waves, chunks that are not whole, the most that is taken; columns that are no
# multiple of a block's)
@pytest.mark.parametrize("M,N,K", [(1, 4096, 1024), (2, 6144, 1024), (8, 6144, 1024), (5, 6272, 1024), (3, 1000, 272), (16, 256, 496), (16, 320, 256),
                                   (7, 512, 1040), (4, 1024, 2048), (2, 192, 4096), (1, 64, 3104)])
def test_norm_in_front(ops, M, N, K):
    g = torch.Generator().manual_seed(M * K + N)
    h, parts = torch.randn(M, K, generator=g).cuda(), torch.randn(2, M, K, generator=g).cuda()
    w = (torch.randn(N, K, generator=g) * K ** -0.5).cuda()
    weight, bias = (1 + 0.1 * torch.randn(K, generator=g)).cuda(), torch.randn(N, generator=g).cuda()
    assert ops.gemm_norm_supported(M, w)
    for delta, b in ((None, None), (parts[:1], bias), (parts, None)):
        stream = h.clone()
        x = ops.rmsnorm(stream, weight, 1e-6, torch.float32, delta=delta)
        want = ops.gemm(x, w, b)
        summed = torch.full_like(h, float("nan")) if delta is not None else None
        got = ops.gemm(h, w, b, norm_weight=weight, norm_eps=1e-6, delta=delta, stream_out=summed)
        assert got.dtype == torch.float32 and torch.equal(got, want)
        if delta is not None:
            assert torch.equal(summed, stream)
        s = (h if delta is None else h + delta.sum(0)).double()
        ref = (s / (s.pow(2).mean(1, keepdim=True) + 1e-6).sqrt() * weight.double()) @ w.double().t() + (0 if b is None else b.double())
        # (K products of a row of order one, each rounded to 2^-24, and the sums' own roundings)
        assert float((got - ref).abs().max()) <= K ** 0.5 * 2.0 ** -22
        if N % 64 == 0 and ops.gemm_silu_supported(h, w):
            want = ops.silu_mul(ops.gemm(x, w, b), interleaved=True)
            got = ops.gemm(h, w, b, norm_weight=weight, norm_eps=1e-6, delta=delta, stream_out=summed, epilogue=ops.EPI_SILU_MUL_IL)
            assert torch.equal(got, want)


@pytest.mark.parametrize("M,N,K", [(1, 64, 16), (16, 128, 80), (13, 6144, 1024), (2, 24576, 4096), (16, 16384, 1040), (8, 12288, 2560), (3, 2048, 4096), (2, 8256, 512)])
def test_silu_behind(ops, M, N, K):
    g = torch.Generator().manual_seed(M + K + N)
    x, w, bias = torch.randn(M, K, generator=g).cuda(), (torch.randn(N, K, generator=g) * K ** -0.5).cuda(), torch.randn(N, generator=g).cuda()
    assert ops.gemm_silu_supported(x, w)
    for b in (None, bias):
        assert torch.equal(ops.gemm(x, w, b, epilogue=ops.EPI_SILU_MUL_IL), ops.silu_mul(ops.gemm(x, w, b), interleaved=True))


@pytest.mark.parametrize("N", [1, 5, 1000, 1024, 1030, 2048, 2052, 4100])
@pytest.mark.parametrize("K", [64, 192, 512, 1024, 1920, 2048, 3072, 4096, 4160])
def test_few_rows_and_many(ops, N, K):
    """A row's sums beside up to sixteen others, by whole chunks where K is some, and beside forty: one order.  Behind w's end is NaN."""
    g = torch.Generator().manual_seed(N + K)
    x, bias = torch.randn(40, K, generator=g).cuda(), torch.randn(N, generator=g).cuda()
    room = torch.full((N * K + 64 * K,), float("nan"), device="cuda")
    room[:N * K] = torch.randn(N * K, generator=g).cuda()
    w = room[:N * K].view(N, K)
    want = ops.gemm(x, w, bias)
    for m in (1, 3, 16):
        assert torch.equal(ops.gemm(x[:m], w, bias), want[:m]), m


@pytest.mark.parametrize("width", [688, 704, 1000, 2736])
@pytest.mark.parametrize("hidden,rows", [(256, 1), (256, 16), (1024, 2), (1024, 8), (240, 3), (1024, 9)])
@pytest.mark.parametrize("bias", [False, True])
def test_a_feed_forward_of_any_width(ops, width, hidden, rows, bias):
    """From the stream, with what is to be added to it, and from rows that the norm's own kernel made: the same bits, also where gate and up
    rows are not interleaved (a width that is no multiple of 32) and where the norm has no room inside the product."""
    from qwen_engine_amd.config import RMSNormSpec, SwiGLUSpec
    from qwen_engine_amd.parts import Runtime, build_part
    from qwen_engine_amd.parts.base import Stream, StreamInput
    g = torch.Generator().manual_seed(width + rows)
    rt = Runtime(torch.device("cuda:0"), torch.float32)
    spec = SwiGLUSpec(intermediate_size=width, bias=True) if bias else SwiGLUSpec(intermediate_size=width)
    ffn, norm = build_part(spec, hidden), build_part(RMSNormSpec(eps=1e-6), hidden)
    ffn.load({n: torch.randn(tuple(t.shape), generator=g) * hidden ** -0.5 for n, t in type(ffn).expected_tensors(spec, hidden).items()}, rt)
    norm.load({"weight": 1 + 0.1 * torch.randn(hidden, generator=g)}, rt)
    assert ffn.interleaved == (width % 32 == 0)
    h, parts = torch.randn(rows, hidden, generator=g).cuda(), torch.randn(2, rows, hidden, generator=g).cuda()
    for delta in (None, parts[0], parts[:1], parts):
        stream = Stream(h.clone(), torch.full_like(h, float("nan")))
        want = ffn.forward(norm.forward(want_h := h.clone(), rt, delta=delta), None)
        x = StreamInput(stream, delta, norm, *norm.fusable_weight(), rt)
        assert x.fusable() and torch.equal(ffn.forward(x, None), want) and torch.equal(stream.h, want_h)


@pytest.mark.parametrize("hidden,rows,heads,kv_heads", [(256, 1, 4, 2), (256, 16, 4, 4), (1024, 2, 16, 8), (1024, 8, 16, 2), (240, 3, 4, 2), (1024, 9, 16, 8)])
@pytest.mark.parametrize("bias", [False, True])
@pytest.mark.parametrize("window", [None, 20])
def test_an_attention_part_of_few_rows(ops, hidden, rows, heads, kv_heads, bias, window):
    """Single tokens, an attention part from the stream with what is to be added to it, and from rows that the norm's own kernel made: the same output, cache
    and stream, also where the norm has no room inside the product."""
    from types import SimpleNamespace
    from qwen_engine_amd.config import AttentionSpec, RMSNormSpec, RopeSpec
    from qwen_engine_amd.parts import Runtime, build_part
    from qwen_engine_amd.parts.base import Stream, StreamInput
    D, P = 64, 16
    g = torch.Generator().manual_seed(hidden + rows + heads)
    rt = Runtime(torch.device("cuda:0"), torch.float32)
    spec = AttentionSpec(heads, kv_heads, D, D ** -0.5, qkv_bias=bias, qk_norm_eps=1e-6, window=window, position=RopeSpec(10000.0, D, 128))
    part, norm = build_part(spec, hidden), build_part(RMSNormSpec(eps=1e-6), hidden)
    part.load({n: torch.randn(tuple(t.shape), generator=g) * hidden ** -0.5 for n, t in type(part).expected_tensors(spec, hidden).items()}, rt)
    norm.load({"weight": 1 + 0.1 * torch.randn(hidden, generator=g)}, rt)
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device="cuda")
    pos = [(11 * i + 5) % 64 for i in range(rows)]
    cache = torch.randn(4 * rows, 2, kv_heads, P, D, generator=g).cuda()
    table = torch.arange(4 * rows, dtype=torch.int32, device="cuda").view(rows, 4)
    ctx = SimpleNamespace(rt=rt, positions=i32(pos), tok_seq=i32(range(rows)), block_tables=[table], shared_keys=None, max_position=max(pos), page_size=P,
                          slots=[i32([(4 * i + p // P) * P + p % P for i, p in enumerate(pos)])], memo={}, num_tokens=rows,
                          extras={type(part): {"dec_tokens": i32(range(rows)), "other_tokens": None, "max_dec_position": max(pos)}})
    bind = lambda kv: SimpleNamespace(kv=kv, group=0, write=True)
    h, parts = torch.randn(rows, hidden, generator=g).cuda(), torch.randn(2, rows, hidden, generator=g).cuda()
    for delta in (None, parts[0], parts[:1], parts):
        stream, one, two = Stream(h.clone(), torch.full_like(h, float("nan"))), cache.clone(), cache.clone()
        want = part.forward(norm.forward(want_h := h.clone(), rt, delta=delta), ctx, bind(two))
        x = StreamInput(stream, delta, norm, *norm.fusable_weight(), rt)
        assert x.fusable() and torch.equal(part.forward(x, ctx, bind(one)), want)
        assert torch.equal(stream.h, want_h) and torch.equal(one, two)


def test_silu_in_the_products_launch(ops):
    """Only where that is not slower: two rows against 24576 x 4096 took 127 us in it, 78 apart."""
    inside = ops.load_library().qe_gemm_f32_silu_inside
    for taken in ((2, 6144, 1024), (16, 1024, 512), (2, 24576, 256), (2, 24576, 1536), (8, 24576, 4096), (8, 8192, 4096)):
        assert inside(*taken) == 1, taken
    for apart in ((2, 24576, 4096), (2, 2048, 4096), (16, 512, 2048), (8, 24576, 2048), (1, 12288, 1024), (2, 6144, 4096)):
        assert inside(*apart) == 0, apart
    assert inside(17, 6144, 1024) == inside(2, 6144, 1000) == inside(2, 24576, 1024) == -1


@pytest.mark.parametrize("M,N,K", [(1, 2000, 1024), (16, 1376, 256), (3, 34, 496)])
def test_norm_in_front_of_gate_and_up_rows(ops, M, N, K):
    g = torch.Generator().manual_seed(M * K + N)
    h, w, weight = torch.randn(M, K, generator=g).cuda(), torch.randn(N, K, generator=g).cuda(), torch.randn(K, generator=g).cuda()
    out = torch.empty(M, N // 2, device="cuda")
    got = ops.gemm(h, w, out=out, epilogue=ops.EPI_SILU_MUL, norm_weight=weight, norm_eps=1e-6)
    assert got is out and torch.equal(got, ops.silu_mul(ops.gemm(ops.rmsnorm(h, weight, 1e-6, torch.float32), w)))
    with pytest.raises(ops.KernelError):
        ops.gemm(h, w, out_dtype=torch.bfloat16, epilogue=ops.EPI_SILU_MUL, norm_weight=weight, norm_eps=1e-6)


@pytest.mark.parametrize("N,K", [(16384, 2048), (16385, 2048), (20000, 1152), (20000, 512)])
def test_few_rows_against_many(ops, N, K):
    """One row goes by rows where two go by chunks: one order."""
    g = torch.Generator().manual_seed(N + K)
    x, w = torch.randn(17, K, generator=g).cuda(), torch.randn(N, K, generator=g).cuda()
    want = ops.gemm(x, w)
    for m in (1, 2, 16):
        assert torch.equal(ops.gemm(x[:m], w), want[:m]), m


def test_what_is_not_taken(ops):
    """More numbers than the norm has room for, rows of no whole steps: refused."""
    w = torch.zeros(64, 1024, device="cuda")
    assert not ops.gemm_norm_supported(9, w) and not ops.gemm_norm_supported(17, w)
    assert not ops.gemm_norm_supported(1, torch.zeros(64, 1032, device="cuda")) and not ops.gemm_norm_supported(1, torch.zeros(64, 240, device="cuda"))
    assert not ops.gemm_silu_supported(torch.zeros(17, 1024, device="cuda"), w)
    with pytest.raises(ops.KernelError):
        ops.gemm(torch.zeros(9, 1024, device="cuda"), w, norm_weight=torch.ones(1024, device="cuda"), norm_eps=1e-6)


def test_matrix_units_switched_off(ops):
    """What goes together on the matrix units is taken apart with them switched off."""
    x, w = torch.zeros(2, 1024, device="cuda"), torch.zeros(4096, 1024, device="cuda")
    qkv, cache = torch.zeros(2, 4096, device="cuda"), torch.zeros(4, 2, 8, 16, 128, device="cuda")
    taken = lambda: (ops.gemm_norm_supported(2, w), ops.gemm_norm_preferred(2, w, 1), ops.gemm_silu_supported(x, w),
                     ops.attention_decode_fused_supported(qkv, cache, 16, None))
    assert taken() == (True,) * 4
    try:
        ops.use_matrix_f32(False)
        assert taken() == (False,) * 4
    finally:
        ops.use_matrix_f32(True)
    assert taken() == (True,) * 4
