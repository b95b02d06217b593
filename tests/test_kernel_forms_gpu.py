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
