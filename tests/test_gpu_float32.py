"""The kernels of the true 32-bit path against float64, and their promise that a result does not depend on what it is computed
beside: every form of a kernel gives the same bits."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


# K: less than a block, several short chunks, chunks that end inside a step, rows that are not on 16 bytes; N: less than a
# tile, one feature past tiles, no multiple of 4; M: the edges of 16, 32, 64 and 128 rows
@pytest.mark.parametrize("K", [3, 96, 130, 1408, 4100])
@pytest.mark.parametrize("M,N", [(1, 5), (16, 64), (17, 129), (33, 77), (64, 4160), (65, 130), (129, 257)])
def test_product_forms_are_one(M, N, K):
    from xinfer_amd import kernels
    g = torch.Generator().manual_seed(M * 7 + N + K)
    x, w = torch.randn(M, K, generator=g), torch.randn(N, K, generator=g)
    xd, wd = x.to(DEV), w.to(DEV)
    ref = x.double() @ w.double().T
    got = {f: kernels.gemm_tn(xd, wd, form=f) for f in ([0, 1] if M <= 64 else []) + [2, 3, 4]}
    y = kernels.gemm_tn(xd, wd)
    for f, v in got.items():
        assert torch.equal(v, y), f
    # a sum of K float32 products in any order: K / 2 roundings of partial sums of about sqrt(k), 2^-24 each, at worst
    bound = 2.0 ** -24 * max(8.0, K ** 0.5) * K ** 0.5
    assert float((y.cpu().double() - ref).abs().max()) < 4 * bound
    r = M // 2
    assert torch.equal(kernels.gemm_tn(xd[r:r + 1].contiguous(), wd)[0], y[r])
    base = torch.randn(M, N, generator=g).to(DEV)
    for f in got:
        acc = base.clone()
        kernels.gemm_tn(xd, wd, out=acc, accumulate=True, form=f)
        assert torch.equal(acc, base + y), f
    if K > 4:           # operands that do not start on 16 bytes
        flat = torch.zeros(M * K + 1, device=DEV)
        flat[1:] = xd.reshape(-1)
        assert torch.equal(kernels.gemm_tn(flat[1:].view(M, K), wd), y)


def test_product_form_refused():
    from xinfer_amd import kernels
    x, w = torch.zeros(65, 32, device=DEV), torch.zeros(8, 32, device=DEV)
    with pytest.raises(kernels.KernelError):
        kernels.gemm_tn(x, w, form=0)
    with pytest.raises(kernels.KernelError):
        kernels.gemm_tn(x, w, form=5)
