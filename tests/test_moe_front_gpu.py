"""Grouped routing by the lanes of a wave, and with the sort in one launch."""
import pytest
import torch

import qwen_engine_amd  # noqa: F401

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.fixture(scope="module")
def ops():
    from qwen_engine_amd.kernels import ops as o
    return o


def _choices(logits, G, keep, top):
    """The same on the host: the lower index first on ties; a row of garbage has scores of zero."""
    E = logits.shape[1]
    ids, weights = [], []
    for z in logits.double():
        p = torch.softmax(z, 0) if not z.isnan().any() else torch.zeros(E, dtype=torch.float64)
        best = p.view(G, -1).max(1).values
        groups = sorted(range(G), key=lambda g: (-float(best[g]), g))[:keep]
        order = sorted((e for e in range(E) if e // (E // G) in groups), key=lambda e: (-float(z[e]) if not z.isnan().any() else 0.0, e))[:top]
        ids.append(order)
        weights.append([float(p[e]) for e in order])
    return ids, torch.tensor(weights)


@pytest.mark.parametrize("E,G,keep,top", [(1, 1, 1, 1), (6, 3, 2, 2), (32, 4, 2, 4), (64, 8, 3, 6), (64, 1, 1, 64), (63, 21, 20, 5), (66, 3, 2, 4)])
@pytest.mark.parametrize("T", [1, 5, 130])
def test_routing_and_its_ties(ops, E, G, keep, top, T):
    g = torch.Generator().manual_seed(E + T)
    logits = torch.randn(T, E, generator=g)
    logits[::3] = torch.randint(-2, 3, (len(logits[::3]), E), generator=g).float()       # (ties)
    if T > 4:
        logits[4] = float("nan")
        logits[3, E // 2] = 60.0               # (beyond 87 above the others, their 32-bit exponentials are all zero, and ties)
    want, weights = _choices(logits, G, keep, top)
    for transposed in (False, True):
        ids, w = ops.moe_route((logits.t().contiguous() if transposed else logits).to(DEV), G, keep, top, transposed=transposed)
        assert ids.tolist() == want
        # (32-bit exponentials and their sum: some 2^-22 of each weight)
        assert (w.cpu().double() - weights).abs().max() <= 1e-6


@pytest.mark.parametrize("T,E,G,keep,top", [(1, 32, 4, 2, 4), (3, 6, 3, 2, 2), (16, 64, 8, 4, 3), (17, 64, 8, 4, 3), (32, 32, 4, 2, 4), (33, 8, 2, 1, 4),
                                           (256, 8, 2, 1, 4), (257, 8, 2, 1, 4)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_experts_with_the_routing_inside(ops, T, E, G, keep, top, dtype):
    """Routing and sort in one launch (up to 32 tokens, and 1024 scores), else apart: the bits that given ids and weights have."""
    g = torch.Generator().manual_seed(T)
    H, F = 64, 32
    x = torch.randn(T, H, generator=g).to(dtype).to(DEV)
    wgu = (torch.randn(E, 2 * F, H, generator=g) / 8).to(dtype).to(DEV)
    wd = (torch.randn(E, H, F, generator=g) / 6).to(dtype).to(DEV)
    logits = torch.randn(T, E, generator=g).to(DEV)
    ids, weights = ops.moe_route(logits, G, keep, top)
    want = ops.moe_experts(x, ids, weights, wgu, wd, 0.8, 1.702, interleaved=True)
    for z, transposed in ((logits, False), (logits.t().contiguous(), True)):
        got = ops.moe_experts(x, None, None, wgu, wd, 0.8, 1.702, interleaved=True, grouped_route=(z, G, keep, top, transposed))
        assert torch.equal(got, want)


def test_many_tokens_are_routed_by_many_blocks(ops):
    """One block takes them only where it is quicker than two launches: 64 tokens of 64 experts took 55 us in it, 34 apart."""
    in_one = ops.load_library().qe_moe_front_grouped_supported
    assert in_one(1, 64, 8) and in_one(16, 64, 6) and in_one(32, 32, 4) and in_one(32, 8, 2)
    assert not (in_one(17, 64, 6) or in_one(33, 8, 2) or in_one(64, 64, 6) or in_one(1, 65, 2))


@pytest.mark.parametrize("kind", ["grouped", "biased", "top_softmax", "sigmoid"])
@pytest.mark.parametrize("T", [64, 65, 300])
def test_a_router_held_in_32_bit(ops, kind, T):
    """Beside bfloat16 rows and experts, with rows enough for the router's product to be turned: what the rows give in portions of 50."""
    from qwen_engine_amd.config import spec as S
    from qwen_engine_amd.parts import Runtime, build_part
    E, H, F = 16, 128, 64
    spec = {"grouped": lambda: S.GroupedMoESpec(num_experts=E, top=4, num_groups=4, keep_groups=2, intermediate_size=F, limit=7.0),
            "biased": lambda: S.BiasedMoESpec(num_experts=E, num_identity=2, top=3, intermediate_size=F, route_scale=1.5),
            "top_softmax": lambda: S.TopSoftmaxMoESpec(num_experts=E, top=4, intermediate_size=F, shared_intermediate_size=96, shared_gate=True),
            "sigmoid": lambda: S.SigmoidMoESpec(num_experts=E, top=2, intermediate_size=F)}[kind]()
    part, rt = build_part(spec, H), Runtime(torch.device(DEV), torch.bfloat16)
    g = torch.Generator().manual_seed(T)
    tensors = {n: torch.randn(tuple(t.shape), generator=g) * H ** -0.5 for n, t in type(part).expected_tensors(spec, H).items()}
    tensors = {n: t if n in ("router", "correction") else t.bfloat16() for n, t in tensors.items()}
    part.load(tensors, rt)
    assert part.w_router.dtype == torch.float32
    from types import SimpleNamespace
    ctx = SimpleNamespace(rt=rt)
    x = torch.randn(T, H, generator=g).bfloat16().to(DEV)
    got = part.forward(x, ctx).sum(0)
    want = torch.cat([part.forward(part_x, ctx).sum(0) for part_x in x.split(50)])
    # (the same logits and choices; the experts' products in other forms, whose sums are rounded to bfloat16 once on the way)
    assert float((got - want).norm() / want.norm()) < 2.0 ** -7
