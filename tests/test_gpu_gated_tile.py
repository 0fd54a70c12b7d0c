"""The feed-forward's first product with its activation in tiles of many rows (`linear_gated_tile`) and the product of a long K in the
lowest tiles that are one round (`linear_tall`) against float64, and the rules that choose them (CPU)."""
import pytest
import torch

from xinfer_amd import kernels

DEV = "cuda:0"


def _last_round(M, F):
    """How the kernel of 256 rows by 128 features takes the tiles behind the last whole round of 256: 1 uncut, 2 in halves of the rows, 4."""
    tiles = -(-M // 256) * -(-F // 128)
    rest = tiles % 256
    return 1 if tiles < 256 or rest == 0 or rest > 128 else 4 if rest <= 64 else 2


def test_every_last_round_is_among_the_sizes():
    """Uncut, halves and quarters all run below, halves and quarters with a last tile of rows that ends in its first half too."""
    marks = [m for m in test_gated_product_in_tiles.pytestmark if m.name == "parametrize"]
    sizes = [(M, F) for M, F, _, _ in marks[0].args[1]]
    assert {_last_round(*s) for s in sizes} == {1, 2, 4}
    assert {_last_round(M, F) for M, F in sizes if 0 < M % 256 <= 128 and M > 256} >= {2, 4}
    assert {_last_round(M, F) for M, F in sizes if M % 256 > 128} >= {2}


@pytest.mark.gpu
@pytest.mark.parametrize("M,F,K,act", [
    (65, 320, 128, "silu"), (1, 4, 64, "gelu_tanh"), (257, 132, 192, "gelu_tanh"), (300, 12288, 64, "silu"),
    (700, 17408, 128, "silu"), (2048, 5000, 64, "gelu_tanh"),
    (1024, 9000, 64, "silu"), (1100, 7168, 64, "gelu_tanh"),
    (2048, 6144, 64, "silu"), (1800, 5300, 128, "gelu_tanh"), (1992, 5300, 64, "silu"), (1800, 4604, 64, "silu")])
def test_gated_product_in_tiles(M, F, K, act):
    g = torch.Generator().manual_seed(M + F)
    x, w = torch.randn(M, K, generator=g).to(torch.bfloat16), (torch.randn(2 * F, K, generator=g) * K ** -0.5).to(torch.bfloat16)
    z = (x.to(DEV).double() @ w.to(DEV).double().t()).cpu()
    a, b = z[:, :F], z[:, F:]
    ref = (torch.nn.functional.silu(a) if act == "silu" else torch.nn.functional.gelu(a, approximate="tanh")) * b
    got = [kernels.linear_gated_tile(x.to(DEV), w.to(DEV), act, shape).cpu() for shape in (0, 1, 2)]
    # one rounding to bfloat16 (8 significant bits, neighbours 2^-7 of a power of two apart: at most 2^-8 of an element); the float32 sums and the activation's exponential add up to
    # (K + 20) 2^-24 of the terms' absolute values, which are below 8 here for sums of K products of unit variance
    bound = 2.0 ** -8 * ref.abs() + 8 * (K + 20) * 2.0 ** -24 * (1 + b.abs() + a.abs())
    assert bool(((got[0].double() - ref).abs() <= bound).all())
    assert torch.equal(got[0], got[1]) and torch.equal(got[0], got[2])


class _Rows:
    """An operand's type, sizes, order and place, all that the rule looks at."""
    dtype = torch.bfloat16

    def __init__(self, *shape, start=0, contiguous=True, dtype=torch.bfloat16):
        self.shape, self.start, self.contiguous, self.dtype = shape, start, contiguous, dtype

    dim = lambda self: len(self.shape)
    data_ptr = lambda self: self.start
    is_contiguous = lambda self: self.contiguous


@pytest.mark.parametrize("M,F,K,shape", [
    (64, 3072, 1024, None), (65, 3072, 1024, 0), (320, 3072, 1024, 0), (321, 3072, 1024, 1), (1280, 3072, 1024, 1),
    (1281, 3072, 1024, 2), (128, 8192, 2048, 0), (129, 8192, 2048, None), (512, 8192, 2048, 1), (513, 8192, 2048, None),
    (897, 8192, 2048, 2), (4096, 12288, 4096, None), (511, 17408, 5120, None), (512, 17408, 5120, 2), (513, 17408, 5120, None),
    (700, 17408, 5120, 2), (2048, 25600, 5120, 2), (2049, 25600, 5120, 2), (256, 3074, 1024, None), (256, 3072, 1000, None),
    # too few workgroups: the library's smaller tiles fill the chip
    (512, 64, 5120, None), (512, 1536, 5120, None), (2048, 2048, 7168, None), (4096, 64, 8192, None), (65, 64, 2048, None),
    (128, 512, 2048, None), (128, 1024, 1088, None), (256, 768, 2048, 0), (65, 64, 1024, 0),
    # the last round: cut, or too much of it, or the library's even rounds at other K
    (1024, 10240, 4608, 2), (1024, 10304, 4608, None), (1024, 12288, 5120, None), (1024, 12288, 4608, None), (1230, 8192, 4160, 2),
    (2048, 8192, 8192, None), (2048, 8192, 6144, None), (2048, 8192, 5120, 2), (2048, 17408, 6144, 2), (2048, 25600, 6144, None),
    (640, 12288, 5120, None), (4096, 8192, 5120, None), (1024, 6144, 5120, None), (1280, 5120, 5120, 2)])
def test_gated_tile_rule(M, F, K, shape):
    """Where the tiled product is taken, and never an operand that it does not take."""
    x, w = _Rows(M, K), _Rows(2 * F, K)
    assert kernels.gated_tile_shape(x, w) == shape
    for other in (_Rows(M, K, start=8), _Rows(M, K, contiguous=False), _Rows(M, K, dtype=torch.float32), _Rows(1, M, K),
                  _Rows(M, K + 64)):
        assert kernels.gated_tile_shape(other, w) is None
    for other in (_Rows(2 * F, K, start=8), _Rows(2 * F, K, dtype=torch.float32), _Rows(2 * F + 1, K)):
        assert kernels.gated_tile_shape(x, other) is None


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", [(97, 260, 64), (1, 4, 128), (333, 516, 192), (1000, 1028, 320), (673, 300, 64)])
def test_product_in_tall_tiles(M, N, K):
    g = torch.Generator().manual_seed(M + N)
    x, w = torch.randn(M, K, generator=g).to(torch.bfloat16).to(DEV), torch.randn(N, K, generator=g).to(torch.bfloat16).to(DEV)
    ref = x.double() @ w.double().t()
    got = [kernels.linear_tall(x, w, rows) for rows in kernels.TALL_SHAPES]
    # one rounding to bfloat16, 2^-8 of an element at most, and K float32 roundings of sums of terms of unit variance (below 8 sqrt(K))
    assert bool(((got[0].double() - ref).abs() <= 2.0 ** -8 * ref.abs() + K * 2.0 ** -24 * 8 * K ** 0.5).all())
    assert all(torch.equal(got[0], y) for y in got[1:])
    assert torch.equal(got[0], kernels.linear_tile(x, w, shape=2))


@pytest.mark.parametrize("M,N,K,rows", [
    (1024, 5120, 17408, None), (1025, 5120, 17408, 96), (1152, 5120, 17408, 96), (1153, 5120, 25600, 128), (1536, 5120, 17408, 128),
    (1537, 5120, 17408, 160), (1760, 5120, 25600, 160), (1761, 5120, 17408, None), (2304, 5120, 17408, None), (2305, 5120, 17408, 224),
    (2688, 5120, 17408, 224), (2689, 5120, 17408, None), (2400, 4868, 17408, 224), (2400, 4864, 17408, None), (1500, 8192, 28672, None),
    # where the library is ahead or was not measured: other widths, and few rows at some K
    (2400, 4612, 17408, None), (1280, 8192, 28672, None), (1400, 6144, 20480, None), (1600, 6144, 20480, None), (1600, 5124, 17408, None),
    (1300, 5120, 16384, None), (1300, 5120, 16448, 128), (1300, 5120, 30720, 128), (1300, 5120, 30784, None), (1100, 5120, 18432, None), (1200, 5120, 18432, 128), (1100, 5120, 17920, 96),
    (1100, 5120, 18944, 96),
    (1100, 4096, 16384, None), (1100, 5120, 16320, None), (1100, 5122, 17408, None), (1100, 5120, 17400, None)])
def test_tall_tile_rule(M, N, K, rows):
    """Where the product is taken (never more than a round of 256 workgroups), and never an operand that it does not take."""
    x, w = _Rows(M, K), _Rows(N, K)
    assert kernels.tall_tile_rows(x, w) == rows
    for other in (_Rows(M, K, start=8), _Rows(M, K, contiguous=False), _Rows(M, K, dtype=torch.float32), _Rows(1, M, K),
                  _Rows(M, K + 64)):
        assert kernels.tall_tile_rows(other, w) is None
    assert kernels.tall_tile_rows(x, _Rows(N, K, start=8)) is None


@pytest.mark.gpu
@pytest.mark.parametrize("k_tiles", [1, 2, 3, 4, 5, 6, 7])
def test_rings_of_unequal_depth(k_tiles):
    """Every walk but those of cut last tiles (below) at fewer tiles of k than its rings have stages, and at their first turns: whole numbers of which
    every partial sum is exact in float32."""
    M, N, K = 260, 520, 64 * k_tiles
    g = torch.Generator().manual_seed(k_tiles)
    x, w = (torch.randint(-4, 5, (n, K), generator=g).to(torch.bfloat16).to(DEV) for n in (M, N))
    ref = x.double() @ w.double().t()
    for shape in (0, 1, 2):
        assert torch.equal(kernels.linear_tile(x, w, partial=True, shape=shape)[0].double(), ref)
    for rows in kernels.TALL_SHAPES:
        assert torch.equal(kernels.linear_tall(x, w, rows), ref.float().to(torch.bfloat16))
    # the gated walks' sums are the same, the first shape's among them: one result for all
    got = [kernels.linear_gated_tile(x, w, "silu", shape) for shape in (0, 1, 2)]
    a, b = ref[:, :N // 2], ref[:, N // 2:]
    want = torch.nn.functional.silu(a) * b
    assert bool(((got[0].double() - want).abs() <= 2.0 ** -8 * want.abs() + 2.0 ** -19 * (1 + (a * b).abs())).all())
    assert torch.equal(got[0], got[1]) and torch.equal(got[0], got[2])


@pytest.mark.gpu
@pytest.mark.parametrize("k_tiles", [1, 3, 5, 7, 11])
@pytest.mark.parametrize("M,N", [(2049, 3716), (2300, 3840), (2290, 5100), (1793, 5888)])
def test_walks_of_cut_last_tiles(M, N, k_tiles):
    """A whole round of tiles of 256 by 128 and up to 64 (in quarters) or 128 more (in halves), past fewer and more tiles of k than the rings of their three walks
    have stages, rows and features past the last tile: bit for bit the sums of the other shapes, whole numbers that are exact."""
    K = 64 * k_tiles
    rest = -(-M // 256) * -(-N // 128) - 256
    assert (0 < rest <= 64) == (N < 4000) and 0 < rest <= 128
    g = torch.Generator().manual_seed(M + k_tiles)
    x, w = (torch.randint(-4, 5, (n, K), generator=g).to(torch.bfloat16).to(DEV) for n in (M, 2 * N))
    cut, low, one = (kernels.linear_gated_tile(x, w, "silu", shape) for shape in (2, 0, 1))
    assert torch.equal(cut, low) and torch.equal(cut, one)
    a, b = (x.double() @ w.double().t()).split(N, 1)
    want = torch.nn.functional.silu(a) * b
    assert bool(((cut.double() - want).abs() <= 2.0 ** -8 * want.abs() + 2.0 ** -19 * (1 + (a * b).abs())).all())


@pytest.mark.parametrize("M,F,K,shape", [
    # a round of 128 rows by 128 features, from 3/4 (K up to 4,096) or 7/8 (up to 6,144) of one on
    (128, 14336, 4096, None), (129, 12288, 4096, 1), (129, 12160, 4096, None), (256, 16384, 4096, 1), (256, 16512, 4096, None), (512, 6144, 2304, 1),
    (512, 7168, 5120, 1), (512, 7040, 5120, None), (512, 8192, 6144, 1), (512, 8192, 6208, None),
    # 256 rows: 0.74 of the rounds' room, whole rounds and one of which the last tiles are cut
    (256, 24576, 2112, None), (379, 16384, 4096, 2), (378, 16384, 4096, None), (700, 12288, 4096, 2), (800, 12288, 4096, None), (2048, 12288, 4096, 2),
    (3584, 12288, 4096, 2), (3585, 12288, 4096, None), (2048, 64, 4096, None), (2048, 2048, 4096, 1),
    (769, 17408, 5120, None), (848, 17408, 5120, None), (849, 17408, 5120, 2), (768, 12288, 5120, 2)])
def test_gated_tile_rule_by_rounds(M, F, K, shape):
    x, w = _Rows(M, K), _Rows(2 * F, K)
    assert kernels.gated_tile_shape(x, w) == shape
    for other in (_Rows(M, K, start=8), _Rows(M, K, contiguous=False), _Rows(M, K, dtype=torch.float32), _Rows(M, K + 64)):
        assert kernels.gated_tile_shape(other, w) is None


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", [(1793, 4092, 5120), (2048, 4096, 6144), (1025, 5764, 5184)])
def test_round_tiles(M, N, K):
    """One full round of tiles of 256 by 128: remainders of rows and features, an odd number of tiles of K."""
    from xinfer_amd import kernels
    assert kernels.round_tiles_ahead(M, N, K)
    g = torch.Generator(device="cuda:0").manual_seed(M)
    x, w = (torch.randn(s, generator=g, device="cuda:0").to(torch.bfloat16) for s in ((M, K), (N, K)))
    y = kernels.linear_bf16(x, w)
    assert torch.equal(y, kernels.linear_tile(x, w, shape=1))
    # float32 sums of K products of about one, 2^-24 of sqrt(K) each step at worst, and one rounding to 8 bits
    ref = x.float() @ w.float().T
    assert float(((y.float() - ref).abs() - ref.abs() * 2.0 ** -8).max()) < K * 2.0 ** -24 * K ** 0.5
