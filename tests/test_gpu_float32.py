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


# M: single blocks whose workgroups have 4, 8, 16, 28 and 48 features, several blocks of rows in the kernel for few rows, tiles of every height; K: one block, an odd number of blocks, chunks that end there
@pytest.mark.parametrize("M,N,K", [(5, 70, 40), (72, 48, 2080), (200, 1024, 96), (300, 640, 1000), (2100, 130, 36),
                                   (380, 6600, 40), (400, 6600, 72), (500, 6600, 40),
                                   (5, 1000, 64), (7, 6150, 96), (20, 1030, 40), (40, 4098, 32), (9, 16500, 40), (30, 16500, 72)])
def test_product_parts(M, N, K):
    """Products of three parts: as near to 64 bits as float32 sums, for operands of unequal size too; a result that has no bound, by an
    operand without one or by a sum past the largest number, is what float32 sums give, and its neighbours are untouched."""
    from xinfer_amd import kernels
    g = torch.Generator().manual_seed(M + N + K)
    x = torch.randn(M, K, generator=g) * torch.exp(torch.randn(K, generator=g) * 2)
    w = torch.randn(N, K, generator=g) * torch.exp(torch.randn(N, 1, generator=g))
    y = kernels.gemm_tn(x.to(DEV), w.to(DEV))
    # every product is off by less than 2^-24 of itself; a chain of a block of 32 a step loses up to 2^-23 a step of what it has
    # reached (the matrix cores cut off), which is at most the sum of the sizes, and the up to eight chunks' sum 2^-24 each
    size = x.double().abs() @ w.double().abs().T
    steps = -(-K // 256)
    assert float(((y.cpu().double() - x.double() @ w.double().T).abs() / size).max()) < (steps + 5) * 2.0 ** -23
    x[0, 1], x[1, 0], x[2, K - 1] = float("inf"), float("nan"), 3.4e38
    w[5, 2], w[N - 1, K - 1] = float("-inf"), 7.0
    x[2, 2] = 0.0                          # (3.4e38 w passes the largest float32 and no float64: beside an inf the two would differ)
    x[M - 1], w[7] = 1e20, -1e20
    z = kernels.gemm_tn(x.to(DEV), w.to(DEV)).cpu()
    want = (x.double() @ w.double().T).float()
    whole = torch.isfinite(want)
    whole[2] = False                       # 3.4e38 rounds to no bfloat16: float32 sums in another order
    assert torch.equal(z.isnan(), want.isnan()) and torch.equal(z[want.isinf()], want[want.isinf()])
    same = whole.clone()
    same[:, 5] = same[:, 7] = same[:, N - 1] = False
    same[[0, 1, M - 1]] = False
    assert torch.equal(z[same], y.cpu()[same])
    near = torch.isfinite(want[2])
    assert bool(((z[2] - want[2]).abs()[near] <= 1e-5 * want[2].abs()[near]).all())
    for f in [2, 3, 4]:
        again = kernels.gemm_tn(x.to(DEV), w.to(DEV), form=f).cpu()
        assert torch.equal(again.nan_to_num(1.5, 2.5, 3.5), z.nan_to_num(1.5, 2.5, 3.5)), f


@pytest.mark.parametrize("M,N,K", [(5, 70, 40), (30, 300, 700), (200, 640, 512), (700, 300, 100)])
@pytest.mark.parametrize("x_size,w_size", [(-100, 0), (-116, 0), (0, -124), (-126, 20), (-136, 30), (-70, -60), (100, -110), (-125, 103), (110, -20)])
def test_small_and_large_operands(M, N, K, x_size, w_size):
    """Operands down to the smallest float32 keep their digits, beside others of any size."""
    from xinfer_amd import kernels
    g = torch.Generator().manual_seed(M + x_size)
    x, w = torch.randn(M, K, generator=g) * 2.0 ** (x_size / 2) * 2.0 ** (x_size / 2), torch.randn(N, K, generator=g) * 2.0 ** w_size
    y, size = kernels.gemm_tn(x.to(DEV), w.to(DEV)).cpu().double(), x.double().abs() @ w.double().abs().T
    # as above, half of the smallest float32 for the result; from 2^104 on a result is a float32 sum of up to K / 8 + 4 products a chunk
    bound = size * ((-(-K // 256) + 5) * 2.0 ** -23 if x_size < 104 else (K / 8 + 12) * 2.0 ** -24) + 2.0 ** -149
    assert bool(((y - x.double() @ w.double().T).abs() < bound).all())


@pytest.mark.parametrize("M,N,K", [(5, 70, 40), (40, 70, 700), (64, 300, 2100)])
def test_results_made_again(M, N, K):
    """Operands near the largest float32, whose parts pass it, beside results that do not: finite, the same bits in every form, and other
    results untouched."""
    from xinfer_amd import kernels
    g = torch.Generator().manual_seed(M + N)
    x, w = torch.randn(M, K, generator=g), torch.randn(N, K, generator=g) * 1e-3
    y = kernels.gemm_tn(x.to(DEV), w.to(DEV))
    big = torch.rand(M, generator=g) < 0.3
    big[0], big[1] = True, False
    at = torch.randint(0, K, (M,), generator=g)
    x[torch.arange(M)[big], at[big]] = 3.4e38          # (rounded to bfloat16: no bound)
    got = [kernels.gemm_tn(x.to(DEV), w.to(DEV), form=f) for f in (-1, 0, 1, 2, 3, 4)]
    assert all(torch.equal(v, got[0]) for v in got)
    want, size = x.double() @ w.double().T, x.double().abs() @ w.double().abs().T
    # (chains of up to K / 8 + 4 sums of the eight chunks, and theirs: 2^-24 of the sum of the sizes each)
    assert bool(got[0].isfinite().all()) and float(((got[0].cpu().double() - want).abs() / size).max()) < (K / 8 + 8) * 2.0 ** -24
    assert torch.equal(got[0][~big.to(DEV)], y[~big.to(DEV)])


@pytest.mark.parametrize("M,N,K", [(8, 4096, 4096), (562, 4096, 4096)])
def test_results_without_a_bound_in_bounded_time(M, N, K):
    """A NaN in every row: a few times a product's time (an element at a time was 40 to 80 times)."""
    from xinfer_amd import kernels

    def time(x):
        for _ in range(2):
            kernels.gemm_tn(x, w)
        a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        a.record()
        for _ in range(5):
            kernels.gemm_tn(x, w)
        b.record()
        torch.cuda.synchronize()
        return a.elapsed_time(b)

    x, w = torch.randn(M, K, device=DEV), torch.randn(N, K, device=DEV)
    plain = time(x)
    x[:, 5] = float("nan")
    assert bool(kernels.gemm_tn(x, w).isnan().all()) and time(x) < 20 * plain


# tiles of 32 and of 64 rows for short K: edges of tiles, one step, an odd number of steps, rows that are not on 16 bytes
@pytest.mark.parametrize("M,N,K", [(3, 5, 16), (33, 70, 3), (700, 1024, 100), (1300, 301, 256), (4097, 4096, 16), (10007, 130, 96), (20000, 129, 1024),
                                   (70001, 65, 33), (5000, 300, 2080)])
def test_short_products(M, N, K):
    from xinfer_amd import kernels
    assert kernels.gemm_f32_form(M, N, K) == 5
    g = torch.Generator(device=DEV).manual_seed(M + N)
    x, w, base = (torch.randn(s, generator=g, device=DEV) for s in ((M, K), (N, K), (M, N)))
    y = kernels.gemm_tn(x, w)
    for f in (2, 3, 4):
        assert torch.equal(kernels.gemm_tn(x, w, form=f), y), f
    size = x.double().abs() @ w.double().abs().T
    assert float(((y.double() - x.double() @ w.double().T).abs() / size).max()) < (-(-K // 256) + 5) * 2.0 ** -23       # as above
    assert torch.equal(kernels.gemm_tn(x, w, out=base.clone(), accumulate=True), base + y)
    flat = torch.zeros(M * K + 1, device=DEV)
    flat[1:] = x.reshape(-1)
    assert torch.equal(kernels.gemm_tn(flat[1:].view(M, K), w), y)
    x[M // 2, K - 1], x[M - 1, 0], w[N - 1, 0] = float("inf"), float("nan"), 3.0
    z, want = kernels.gemm_tn(x, w), x.double() @ w.double().T
    assert torch.equal(z.isnan(), want.isnan()) and torch.equal(z.isposinf(), want.isposinf()) and torch.equal(z.isneginf(), want.isneginf())
    others = torch.arange(M, device=DEV)[(torch.arange(M, device=DEV) != M // 2) & (torch.arange(M, device=DEV) != M - 1)]
    assert torch.equal(z[others][:, :N - 1], y[others][:, :N - 1])


@pytest.mark.parametrize("M,N,K", [(4096, 16, 4096), (10007, 16, 1024), (4096, 128, 1024), ((1 << 24) + 5, 3, 4)])
def test_many_rows_of_few_features(M, N, K):
    """The kernel for few rows over many blocks of rows, on all dies; more rows than its workgroups make a launch."""
    from xinfer_amd import kernels
    assert kernels.gemm_f32_form(M, N, K) < 2 or M > 1 << 20
    g = torch.Generator(device=DEV).manual_seed(N)
    x, w = torch.randn(M, K, generator=g, device=DEV), torch.randn(N, K, generator=g, device=DEV)
    y = kernels.gemm_tn(x, w)
    size = x.double().abs() @ w.double().abs().T
    assert float(((y.double() - x.double() @ w.double().T).abs() / size).max()) < (-(-K // 256) + 5) * 2.0 ** -23
    if M < 1 << 20:
        assert torch.equal(kernels.gemm_tn(x, w, form=2), y)
    assert torch.equal(kernels.gemm_tn(x[-50:], w), y[-50:])


# I: one tile, one feature past four, walks of one to three tiles with short last ones; K: no multiple of 4, chunks that end inside a step
@pytest.mark.parametrize("I,K", [(40, 4100), (17, 130), (1000, 96), (3072, 1024), (4090, 257), (8190, 64), (12288, 72)])
@pytest.mark.parametrize("M", [1, 7, 16])
def test_gated_product_is_the_two_kernels(M, I, K):
    """Gate, up and silu(gate) * up in one pass: the bits of the product and the activation behind it, operands without a bound among them."""
    from xinfer_amd import kernels
    g = torch.Generator().manual_seed(M + I + K)
    x, w = torch.randn(M, K, generator=g).to(DEV), (torch.randn(2 * I, K, generator=g) * 2 * K ** -0.5).to(DEV)
    assert kernels.gemm_gated_rows(I, K) >= M
    assert torch.equal(kernels.gemm_gated(x, w), kernels.silu_mul(kernels.gemm_tn(x, w)))
    flat = torch.zeros(M * K + 1, device=DEV)          # x not on 16 bytes
    flat[1:] = x.reshape(-1)
    assert torch.equal(kernels.gemm_gated(flat[1:].view(M, K), w), kernels.silu_mul(kernels.gemm_tn(x, w)))
    w[I - 1, 0], w[2 * I - 1, 1], w[I, K - 1] = float("inf"), float("nan"), 3.4e38
    x[M - 1, 2] = float("-inf")
    got, want = kernels.gemm_gated(x, w), kernels.silu_mul(kernels.gemm_tn(x, w))
    assert torch.equal(got.nan_to_num(1.5, 2.5, 3.5), want.nan_to_num(1.5, 2.5, 3.5)) and torch.equal(got.isnan(), want.isnan())


def test_gated_product_refused():
    """More rows than go in the kernel for few rows, and outputs with an empty last round of workgroups: the two kernels."""
    from xinfer_amd import kernels
    assert kernels.gemm_gated_rows(17408, 5120) == 0 and kernels.gemm_gated_rows(0, 64) == 0
    with pytest.raises(kernels.KernelError):
        kernels.gemm_gated(torch.zeros(17, 64, device=DEV), torch.zeros(64, 64, device=DEV))
    with pytest.raises(kernels.KernelError):
        kernels.gemm_gated(torch.zeros(4, 64, device=DEV), torch.zeros(65, 64, device=DEV))


def test_product_form_refused():
    from xinfer_amd import kernels
    x, w = torch.zeros(65, 32, device=DEV), torch.zeros(8, 32, device=DEV)
    with pytest.raises(kernels.KernelError):
        kernels.gemm_tn(x, w, form=0)
    with pytest.raises(kernels.KernelError):
        kernels.gemm_tn(x, w, form=5)


def _plain_attention(q, k, v, scale, window, chunk, cap, slopes, sinks):
    """q [T, H, d] at the last T of the positions of k [L, G, d], v [L, G, dv]; float64."""
    T, H, L = q.shape[0], q.shape[1], k.shape[0]
    i, j = torch.arange(L - T, L)[:, None], torch.arange(L)[None]
    seen = j <= i
    if window:
        seen = seen & (i - j < window)
    if chunk:
        seen = seen & (i // chunk == j // chunk)
    out = []
    for h in range(H):
        g = h // (H // k.shape[1])
        s = (q[:, h] @ k[:, g].T) * scale
        s = cap * torch.tanh(s / cap) if cap else s
        if slopes is not None:
            s = s - slopes[h] * (i - j)
        s = s.masked_fill(~seen, float("-inf"))
        z = sinks[h].reshape(1, 1).expand(T, 1) if sinks is not None else torch.full((T, 1), float("-inf"), dtype=s.dtype)
        w = torch.softmax(torch.cat([s, z], dim=1), dim=1)[:, :L]
        out.append(torch.where(seen, w, 0.0) @ v[:, g].nan_to_num(0.0, 0.0, 0.0) if window else w @ v[:, g])
    return torch.stack(out, dim=1)


@pytest.mark.parametrize("nq,nkv,d,dv,page,window,chunk,cap,slopes,sinks,latent", [
    (4, 2, 16, 16, 8, 0, 0, 0.0, False, False, False), (6, 2, 48, 80, 16, 0, 0, 0.0, False, False, False),
    (8, 2, 128, 128, 64, 33, 0, 0.0, False, True, False), (17, 1, 64, 112, 16, 0, 40, 5.0, False, True, False),
    (4, 4, 96, 32, 12, 0, 0, 3.0, True, False, False), (40, 1, 256, 192, 64, 0, 0, 0.0, False, True, True),
    (2, 1, 208, 256, 32, 100, 64, 0.0, False, False, False)])
def test_attention(nq, nkv, d, dv, page, window, chunk, cap, slopes, sinks, latent):
    """Portions and single tokens of two requests against float64, every token's bits alone and in the step, and beside the kernel
    for every size; outside the window the first request's keys and values are undefined and must stay unread."""
    from xinfer_amd import kernels
    g = torch.Generator().manual_seed(d + dv)
    lens, news = [300, 41], [37, 41]
    pages = [-(-n // page) for n in lens]
    perm = torch.randperm(sum(pages) + 2, generator=g).tolist()
    bt = torch.zeros(2, max(pages) + 1, dtype=torch.int32)
    kc = torch.full((len(perm), nkv, page, d), float("nan"))
    vc = kc if latent else torch.full((len(perm), nkv, page, dv), float("nan"))
    scale, qs, want = d ** -0.5, [], []
    sl = torch.rand(nq, generator=g) * 0.1 if slopes else None
    sk = torch.randn(nq, generator=g) if sinks else None
    dbl = lambda t: None if t is None else t.double()
    for b, (n, new) in enumerate(zip(lens, news)):
        k = torch.randn(n, nkv, d, generator=g)
        v = k[..., :dv] if latent else torch.randn(n, nkv, dv, generator=g)
        qb = torch.randn(new, nq, d, generator=g) * 2
        qs.append(qb)
        want.append(_plain_attention(qb.double(), k.double(), v.double(), scale, window, chunk, cap, dbl(sl), dbl(sk)))
        first = n - new + 1 - window if window and b == 0 else 0       # what no query of this step sees
        for i in range(n):
            p = perm[sum(pages[:b]) + i // page]
            bt[b, i // page] = p
            if i >= first:
                kc[p, :, i % page] = k[i]
                if not latent:
                    vc[p, :, i % page] = v[i]
    q = torch.cat(qs)
    tok_seq = torch.tensor([b for b in range(2) for _ in range(news[b])], dtype=torch.int32)
    pos = torch.tensor([lens[b] - news[b] + i for b in range(2) for i in range(news[b])], dtype=torch.int32)
    dev = [t.to(DEV) for t in (q, kc, bt, tok_seq, pos)]
    vd = None if latent else vc.to(DEV)
    opt = dict(softcap=cap, slopes=None if sl is None else sl.to(DEV), sinks=None if sk is None else sk.to(DEV),
               value_dim=dv if latent else None, chunk=chunk)
    run = lambda rows, **kw: kernels.attention_generic(dev[0][rows].contiguous(), dev[1], vd, dev[2], dev[3][rows].contiguous(),
                                                       dev[4][rows].contiguous(), scale, window, **opt, **kw)
    assert kernels.lib().xi_attention_f32_takes(nq, nkv, d, dv)
    got = run(slice(None))
    ref = torch.cat(want).reshape(q.shape[0], -1)
    # scores of about 2 whose float32 sums of d products are off by about 2^-24 sqrt(d) of their size, weighed sums likewise
    assert float((got.cpu().double() - ref).abs().max()) < 2e-5
    for r in (0, 20, 36, 37, 77):
        assert torch.equal(run(slice(r, r + 1))[0], got[r]), r
    plain = run(slice(None), matrix=False)
    assert float((plain.cpu().double() - ref).abs().max()) < 2e-5


def test_attention_keys_without_weight():
    """Scores of -inf through whole blocks of keys, at the request's start and further on: no weight for these keys, and
    results undefined only for a token that has no other key."""
    from xinfer_amd import kernels
    g = torch.Generator().manual_seed(5)
    L, nq, nkv, d = 300, 4, 2, 64
    q, k, v = torch.randn(L, nq, d, generator=g), torch.randn(L, nkv, d, generator=g), torch.randn(L, nkv, d, generator=g)
    q[..., 0] = q[..., 0].abs() + 0.1
    off = torch.zeros(L, dtype=torch.bool)
    off[:20] = off[128:160] = True           # wave 0's first block and the second one of waves 0 and 1; a part of wave 1's first
    k[off, :, 0] = float("-inf")
    want = _plain_attention(q.double(), k.double(), v.double(), d ** -0.5, 0, 0, 0.0, None, None)
    pages = lambda x: torch.nn.functional.pad(x, (0, 0, 0, 0, 0, 4)).view(-1, 16, nkv, x.shape[2]).transpose(1, 2).contiguous().to(DEV)
    bt = torch.arange(19, dtype=torch.int32, device=DEV)[None]
    pos = torch.arange(L, dtype=torch.int32, device=DEV)
    for rows in (slice(0, L), slice(20, 21), slice(130, 131), slice(170, 171)):
        got = kernels.attention_generic(q[rows].contiguous().to(DEV), pages(k), pages(v), bt, torch.zeros_like(pos[rows]), pos[rows].contiguous(),
                                        d ** -0.5).cpu().double().view(-1, nq, d)
        has = torch.arange(L)[rows] >= 20
        assert bool(got[~has].isnan().all())
        # as in `test_attention`
        assert float((got[has] - want[rows][has]).abs().max()) < 2e-5, rows


@pytest.mark.parametrize("nq,nkv,d", [(3, 3, 32), (4, 2, 144), (20, 1, 64)])
def test_attention_tiles_are_one(nq, nkv, d):
    """Single tokens and portions side by side: the same bits for every number of tokens a workgroup, tiles where requests meet among
    them, and a request's infinite values stay its own."""
    from xinfer_amd import kernels
    g = torch.Generator().manual_seed(d)
    lens, news = [70, 1, 290, 33, 61, 200], [1, 1, 1, 20, 61, 15]
    mp, page = 10, 32
    kc, vc = (torch.randn(6 * mp, nkv, page, d, generator=g).to(DEV) for _ in range(2))
    bt = torch.randperm(6 * mp, generator=g).to(torch.int32).view(6, mp).to(DEV)
    q = torch.randn(sum(news), nq, d, generator=g).to(DEV)
    seq = torch.tensor([b for b in range(6) for _ in range(news[b])], dtype=torch.int32)
    pos = torch.tensor([lens[b] - news[b] + i for b in range(6) for i in range(news[b])], dtype=torch.int32)
    run = lambda **kw: kernels.attention_generic(q, kc, vc, bt, seq.to(DEV), pos.to(DEV), d ** -0.5, **kw).cpu()
    most = 16 // min(16, nq // nkv)
    want = run(tile=1)
    assert float((want - run(matrix=False)).abs().max()) < 2e-5           # as in `test_attention`
    for tile in range(0, most + 1):
        for lead in (0, 3):
            assert torch.equal(run(tile=tile, lead=lead), want), (tile, lead)
    vc[bt[4].long()] = float("inf")
    vc[bt[2, 1].long()] = float("nan")
    own = (seq == 4) | (seq == 2)
    for tile in {1, most // 2 or 1, most}:
        for lead in (0, 3):
            assert torch.equal(run(tile=tile, lead=lead)[~own], want[~own]), (tile, lead)
    with pytest.raises(kernels.KernelError):
        run(tile=most + 1)
    with pytest.raises(kernels.KernelError):
        run(lead=q.shape[0] + 1)


@pytest.mark.parametrize("page,window,d,news", [(16, 0, 64, 5), (24, 0, 128, 3), (64, 9000, 128, 4), (40, 130, 32, 4), (16, 0, 144, 2)])
def test_attention_past_a_waves_pages(page, window, d, news):
    """Contexts around the 8,192 keys whose pages a wave asks for at once, with pages of whole blocks of 16 keys and others: tokens by
    themselves and in tiles give the same bits, and those of the kernel for every size but for the sums' order."""
    from xinfer_amd import kernels
    g = torch.Generator().manual_seed(page + d)
    lens, nq, nkv = [8192, 8207, 16500, 129], 4, 2
    mp = -(-max(lens) // page)
    kc, vc = (torch.randn(4 * mp, nkv, page, d, generator=g).to(DEV) for _ in range(2))
    bt = torch.randperm(4 * mp, generator=g).to(torch.int32).view(4, mp).to(DEV)
    q = torch.randn(4 * news, nq, d, generator=g).to(DEV)
    seq = torch.arange(4, dtype=torch.int32).repeat_interleave(news).to(DEV)
    pos = torch.tensor([n - news + i for n in lens for i in range(news)], dtype=torch.int32, device=DEV)
    run = lambda **kw: kernels.attention_generic(q, kc, vc, bt, seq, pos, d ** -0.5, window, **kw).cpu()
    one = run(tile=1)
    assert float((one - run(matrix=False)).abs().max()) < 2e-5           # as in `test_attention`
    assert torch.equal(run(tile=min(8, news + 1)), one)
    assert torch.equal(run(tile=8, lead=1), one)


@pytest.mark.parametrize("nq,nkv,d", [(12, 4, 80), (6, 1, 96), (8, 8, 112), (6, 2, 128)])
def test_attention_sizes_between_64_and_128(nq, nkv, d):
    """Head sizes with kernels of their own: tokens by themselves (few and many workgroups) and in tiles the same bits, and those of one lane a key
    but for the sums' order; the same keys with fewer value dims, which go in the kernel with tests, give those dims' bits."""
    from xinfer_amd import kernels
    g = torch.Generator().manual_seed(d)
    lens, news, page = [33, 200, 64, 17] + [130] * 40, [5, 37, 64, 1] + [1] * 40, 16
    mp = -(-max(lens) // page)
    kc, vc = (torch.randn(len(lens) * mp, nkv, page, d, generator=g).to(DEV) for _ in range(2))
    bt = torch.randperm(len(lens) * mp, generator=g).to(torch.int32).view(len(lens), mp).to(DEV)
    q = torch.randn(sum(news), nq, d, generator=g).to(DEV)
    seq = torch.arange(len(lens), dtype=torch.int32).repeat_interleave(torch.tensor(news)).to(DEV)
    pos = torch.tensor([n - new + i for n, new in zip(lens, news) for i in range(new)], dtype=torch.int32, device=DEV)
    run = lambda v, rows=slice(None), **kw: kernels.attention_generic(q[rows].contiguous(), kc, v, bt, seq[rows].contiguous(), pos[rows].contiguous(),
                                                                      d ** -0.5, **kw)
    one = run(vc, tile=1)
    assert float((one - run(vc, matrix=False)).abs().max()) < 2e-5           # as in `test_attention`
    assert torch.equal(run(vc, tile=2), one) and torch.equal(run(vc), one)
    assert torch.equal(run(vc, slice(0, 8)), one[:8]) and torch.equal(run(vc, slice(106, 112)), one[106:112])
    less = run(vc[..., :d - 16].contiguous(), tile=1)
    assert torch.equal(less.view(-1, nq, d - 16), one.view(-1, nq, d)[..., :d - 16])
