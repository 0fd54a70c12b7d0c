"""Products of a round of low tiles (`linear_tile` shapes 7 to 9) against exact sums, and the rule that chooses them (CPU)."""
import pytest
import torch

from xinfer_amd import kernels

DEV = "cuda:0"


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,k_tiles,slices", [(1, 4, 1, 1), (63, 60, 2, 1), (64, 64, 8, 2), (65, 68, 9, 1), (127, 132, 7, 3), (129, 260, 17, 4), (200, 516, 20, 5),
                                                (17, 1024, 33, 8), (130, 124, 48, 12)])
def test_low_tiles(M, N, k_tiles, slices):
    """Rows and features past the last tile, fewer tiles of k than a ring has stages and more, slices a tile apart: whole numbers whose sums are exact."""
    K = 64 * k_tiles
    g = torch.Generator().manual_seed(M + N)
    x, w = (torch.randint(-4, 5, (n, K), generator=g).to(torch.bfloat16).to(DEV) for n in (M, N))
    ref = x.double() @ w.double().t()
    for shape in (7, 8, 9):
        y = kernels.linear_tile(x, w, slices, partial=True, shape=shape)
        assert y.shape == (slices, M, N) and torch.equal(y.double().sum(0), ref)
        for s in range(slices):
            lo, hi = 64 * (s * k_tiles // slices), 64 * ((s + 1) * k_tiles // slices)
            assert torch.equal(y[s].double(), x[:, lo:hi].double() @ w[:, lo:hi].double().t())
        assert torch.equal(kernels.linear_tile(x, w, shape=shape), ref.float().to(torch.bfloat16))


@pytest.mark.gpu
@pytest.mark.parametrize("M", [17, 65, 129, 257, 600])
def test_linear_takes_them(M):
    """... and a weight off 16 bytes goes where it went before."""
    g = torch.Generator().manual_seed(M)
    N, K = 1024, 1024
    x, w = torch.randn(M, K, generator=g).to(torch.bfloat16).to(DEV), (torch.randn(N, K, generator=g) / 32).to(torch.bfloat16).to(DEV)
    ref = x.double() @ w.double().t()
    # a rounding to bfloat16, 2^-8 of an element, and K float32 roundings of sums below 8 in absolute value
    bound = 2.0 ** -8 * ref.abs() + K * 2.0 ** -24 * 8
    for split in (False, True):
        plan = kernels.small_tile_plan(M, N, K, split)
        y = kernels.linear_bf16(x, w, allow_split=split)
        assert y.shape == ((plan[1], M, N) if plan and plan[1] > 1 else y.shape)
        total = y.double().sum(0) if y.dim() == 3 else y.double()
        assert bool(((total - ref).abs() <= bound).all())
    if M > kernels.MID_BLOCK:
        off = torch.empty(N * K + 1, dtype=torch.bfloat16, device=DEV)[1:].view(N, K).copy_(w)
        assert off.data_ptr() % 16
        assert bool(((kernels.linear_bf16(x, off).double() - ref).abs() <= bound).all())


@pytest.mark.parametrize("split", [False, True])
def test_low_tiles_are_one_round(split):
    sizes = [(N, K) for N in (256, 512, 640, 1024, 1000, 2048, 4096, 4384, 6144, 10240, 16768, 24576, 151936) for K in (64, 512, 1000, 1024, 2048, 4096, 12288, 25600)]
    taken = 0
    for N, K in sizes:
        for M in (1, 16, 17, 64, 65, 128, 129, 200, 256, 257, 512, 700, 1024, 1025, 2048, 2049, 5000):
            plan = kernels.small_tile_plan(M, N, K, split)
            if plan is None:
                continue
            taken += 1
            rows, features = {7: (64, 64), 8: (64, 128), 9: (128, 128)}[plan[0]]
            assert -(-M // rows) * -(-N // features) * plan[1] <= kernels.COMPUTE_UNITS and kernels.linear_tile_takes(M, N, K, plan[1])
            assert 17 <= M <= 2048 and (split or plan[1] == 1) and (plan[1] == 1 or K // 64 // plan[1] >= 4)
            assert not split or M > 128 or (N >= 1024 and N * K < 1 << 23)
    assert taken > 50
    plan = kernels.small_tile_plan
    assert plan(256, 4096, 1024, True) == (7, 1) and plan(256, 1024, 2048, True) == (7, 4) and plan(61, 1024, 4096, True) == (7, 11) and plan(40, 4096, 2048, True) is None and plan(61, 4096, 4096, True) is None
    assert plan(256, 10240, 5120, True) is None and plan(256, 5120, 25600, True) is None and plan(2048, 4096, 4096, True) is None
    assert plan(512, 2048, 6144, True) == (9, 4) and plan(768, 2048, 8192, True) is None and plan(512, 4096, 8192, True) is None and plan(256, 1024, 3072, False) is None


SPLIT_SIZES = [(N, K) for N in (1024, 1500, 1536, 2048, 3072, 4096, 6144, 8192, 16768, 32768) for K in (64, 192, 512, 1024, 1536, 2048, 3072, 4096, 5632, 8128)]


def test_sums_of_decode_rows_do_not_follow_the_batch():
    """17 to 128 rows with partial sums: whether a product goes to the low tiles, and in how many slices of K, follows from (N, K) alone."""
    taken = 0
    for N, K in SPLIT_SIZES:
        plans = [kernels.small_tile_plan(M, N, K, True) for M in range(17, 129)]
        assert len({None if p is None else p[1] for p in plans}) == 1, (N, K)
        taken += plans[0] is not None
    assert taken > 20


@pytest.mark.gpu
@pytest.mark.parametrize("N,K", [(1024, 3072), (4096, 1024), (1536, 3584), (1536, 4096), (1028, 1024), (640, 2560)])
def test_a_row_beside_others(N, K):
    """... and so a row's partial sums are the same bits beside 16 others and beside 127."""
    g = torch.Generator().manual_seed(N)
    x, w = torch.randn(128, K, generator=g).to(torch.bfloat16).to(DEV), torch.randn(N, K, generator=g).to(torch.bfloat16).to(DEV)
    y = kernels.linear_bf16(x, w, allow_split=True)
    for M in (17, 32, 37, 64, 65, 66, 100, 127):
        assert torch.equal(kernels.linear_bf16(x[:M].contiguous(), w, allow_split=True), y[:, :M])


def test_whole_products_where_they_are_ahead():
    """No gaps between rows at which nothing was measured behind, and nothing where it was."""
    plan = kernels.small_tile_plan
    for N, M in ((1024, 1024), (2048, 1024), (4096, 512)):
        assert all(plan(m, N, 1024, False) is not None for m in range(32, M + 1))
    for M, N, K in ((493, 6144, 4096), (512, 6144, 4096), (512, 6144, 2560), (512, 7168, 5120), (384, 8192, 1280), (400, 8192, 1024)):
        assert plan(M, N, K, False) is None and plan(M, N, K, M > 256) is None
    for N in (512, 1024):
        assert all(plan(m, N, K, False) is None for m in (32, 64, 128, 256) for K in (1152, 1280))
    assert plan(960, 4096, 2048, False) == (9, 1) and plan(96, 3072, 1152, False) is not None and plan(300, 10240, 1024, False) == (9, 1)
