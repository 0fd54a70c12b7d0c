"""The experts' products in tiles of many rows (`moe_experts_tiled`) against float64, and bit for bit beside the grouped form for
few rows: experts with no row, one row, and rows at the edges of a tile; features and widths that end inside a tile."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _plain(x, gate_up, down, idx, wt, act, gated, weigh_input, E, add):
    x, gate_up, down, wt = x.double(), gate_up.double(), down.double(), wt.double()
    F = gate_up.shape[1] // 2 if gated else gate_up.shape[1]
    f = {"silu": torch.nn.functional.silu, "relu2": lambda z: torch.relu(z) ** 2,
         "gelu_tanh": lambda z: torch.nn.functional.gelu(z, approximate="tanh")}[act]
    out = torch.zeros_like(x)
    for r in range(idx.shape[1]):
        for e in range(int(idx.max()) + 1):
            rows = (idx[:, r] == e).nonzero()[:, 0]
            if not len(rows):
                continue
            w = wt[rows, r, None]
            h = x[rows] * w if weigh_input else x[rows]
            if e >= E:
                y = h
            else:
                u = h @ gate_up[e].T
                u = f(u[:, :F]) * u[:, F:] if gated else f(u)
                y = u @ down[e].T
            out[rows] += y if weigh_input else y * w
    return out if add is None else out + add.double()


@pytest.mark.parametrize("H,F,act,gated,weigh,identity,shared", [
    (64, 64, "silu", True, False, 2, True), (192, 320, "gelu_tanh", True, True, 0, False), (320, 192, "relu2", False, False, 0, True),
    (512, 256, "silu", False, False, 1, False), (256, 576, "silu", True, False, 0, False)])
def test_experts_in_tiles(H, F, act, gated, weigh, identity, shared, monkeypatch):
    from xinfer_amd import kernels
    g = torch.Generator().manual_seed(H + F)
    E, rows = 6, [0, 1, 127, 128, 129, 300]              # pairs an expert (the identity experts take some of the rest)
    rb = lambda *s: torch.randn(*s, generator=g).to(torch.bfloat16)
    gate_up, down = rb(E, (2 if gated else 1) * F, H) * H ** -0.5, rb(E, H, F) * F ** -0.5
    pairs = [e for e, n in enumerate(rows) for _ in range(n)] + [E + i % max(1, identity) for i in range(40) if identity]
    pairs += [5] * (len(pairs) % 2)
    idx = torch.tensor(pairs)[torch.randperm(len(pairs), generator=g)].view(-1, 2).to(torch.int32)
    T = idx.shape[0]
    x, wt = rb(T, H), torch.rand(T, 2, generator=g) + 0.1
    add = rb(T, H) if shared else None
    dev = [t.to(DEV) for t in (x, gate_up, down, idx, wt)]
    kw = dict(gated=gated, weigh_input=weigh, identity=identity, add=None if add is None else add.to(DEV))
    ref = _plain(x, gate_up, down, idx.long(), wt, act, gated, weigh, E, add)
    few = kernels.moe_experts(*dev, act, grouped=True, tile_rows=32, **kw)
    for bm in (64, 128, 256):
        got = kernels.moe_experts_tiled(*dev, act, tile_rows=bm, **kw)
        # one rounding of the hidden rows to bfloat16 (2^-9 of each), averaged over F products
        assert float((got.cpu().double() - ref).norm() / ref.norm()) < 2.0 ** -8
        assert torch.equal(got, few), bm
    assert torch.equal(kernels.moe_experts_tiled(*dev, act, **kw), few)
    for pair in ((256, 128), (128, 256), (256, 64), (64, 128)):          # the products in tiles of their own
        monkeypatch.setattr(kernels, "moe_tile_rows", lambda *a: pair)
        assert torch.equal(kernels.moe_experts_tiled(*dev, act, **kw), few), pair


@pytest.mark.parametrize("H,F,act,gated,weigh,identity", [
    (64, 64, "silu", True, False, 2), (192, 320, "gelu_tanh", True, True, 0), (320, 192, "relu2", False, False, 1), (1088, 576, "silu", True, False, 0),
    (512, 2112, "silu", False, False, 0)])
def test_tiles_of_few_rows(H, F, act, gated, weigh, identity):
    """Tiles of up to 16 rows: the bits of the higher ones, for rows at the edges of a tile and more tiles an expert than there should be."""
    from xinfer_amd import kernels
    g = torch.Generator().manual_seed(H + F)
    rb = lambda *s: torch.randn(*s, generator=g).to(torch.bfloat16)
    for rows in ([0, 1, 15, 16, 17, 33], [0, 0, 2, 0, 0, 0], [3] * 6):
        E = len(rows)
        gate_up, down = rb(E, (2 if gated else 1) * F, H) * H ** -0.5, rb(E, H, F) * F ** -0.5
        pairs = [e for e, n in enumerate(rows) for _ in range(n)] + [E + i % max(1, identity) for i in range(6) if identity]
        idx = torch.tensor(pairs)[torch.randperm(len(pairs), generator=g)].view(-1, 2).to(torch.int32)
        T = idx.shape[0]
        dev = [t.to(DEV) for t in (rb(T, H), gate_up, down, idx, torch.rand(T, 2, generator=g) + 0.1)]
        kw = dict(gated=gated, weigh_input=weigh, identity=identity, add=rb(T, H).to(DEV))
        want = kernels.moe_experts_tiled(*dev, act, tile_rows=64, **kw)
        assert torch.equal(kernels.moe_experts_tiled(*dev, act, tile_rows=16, **kw), want), rows
    assert kernels.moe_tile_rows(8 * E, E, F, H, gated) == (16, 16) and kernels.moe_tile_rows(8 * E + 1, E, F, H, gated) == (64, 64)


@pytest.mark.parametrize("H,F,act,gated", [(2112, 1088, "silu", True), (192, 2112, "relu2", False)])
def test_heights_from_the_counts(H, F, act, gated, monkeypatch):
    """Tiles whose heights are chosen on the device, at the edges of every walk, with columns that do and do not share out over the dies."""
    from xinfer_amd import kernels
    g = torch.Generator(device=DEV).manual_seed(H)
    monkeypatch.setattr(kernels, "moe_tile_rows", lambda *a: (0, 0))
    rb = lambda *s: torch.randn(*s, generator=g, device=DEV).to(torch.bfloat16)
    edges = [0, 1, 64, 65, 128, 129, 160, 161, 192, 193, 224, 225, 256, 257, 511, 700]
    for counts in (edges, [1] * 16, [0, 2000, 0, 1] * 4, [300] * 16):
        E = len(counts)
        gate_up, down = rb(E, (2 if gated else 1) * F, H) * H ** -0.5, rb(E, H, F) * F ** -0.5
        pairs = torch.tensor([e for e, n in enumerate(counts) for _ in range(n)] + [3] * (sum(counts) % 2), device=DEV)
        idx = pairs[torch.randperm(len(pairs), generator=g, device=DEV)].view(-1, 2).to(torch.int32)
        x, wt = rb(idx.shape[0], H), torch.rand(idx.shape, generator=g, device=DEV)
        few = kernels.moe_experts(x, gate_up, down, idx, wt, act, grouped=True, tile_rows=32, gated=gated)
        assert torch.equal(kernels.moe_experts_tiled(x, gate_up, down, idx, wt, act, gated=gated), few), counts


@pytest.mark.parametrize("T,H", [(1, 64), (5, 192), (300, 128)])
def test_the_opened_branch_and_pairs_of_rows(T, H):
    """The branch that a factor opens, added by the pass that adds the experts up or behind it; two scaled rows in one pass or in two:
    the same bits, also for rows that start on any element."""
    from xinfer_amd import kernels
    g = torch.Generator().manual_seed(T + H)
    E, F = 4, 64
    rb = lambda *s: torch.randn(*s, generator=g).to(torch.bfloat16).to(DEV)
    up, down, x = rb(E, F, H), rb(E, H, F), rb(T, H)
    idx, wt = torch.randint(0, E, (T, 2), generator=g).to(torch.int32).to(DEV), torch.rand(T, 2, generator=g).to(DEV)
    extra = (torch.randn(T, 3, generator=g) * 4).to(DEV)
    flat = torch.zeros(T * H + 1, dtype=torch.bfloat16, device=DEV)
    flat[1:] = rb(T * H)
    for add in (rb(T, H), flat[1:].view(T, H)):
        for opening in (extra[:, 1], extra[:, 0].contiguous()):
            got = kernels.moe_experts_tiled(x, up, down, idx, wt, "relu2", gated=False, add=add, opening=opening)
            want = kernels.gated_add_(kernels.moe_experts_tiled(x, up, down, idx, wt, "relu2", gated=False), add, opening)
            assert torch.equal(got, want)
        for a, b in ((x, add), (add, x), (x[:, 1:].contiguous(), add[:, 1:].contiguous()), (x.float(), add.float())):
            assert torch.equal(kernels.scaled_pair(a, 0.75, b, -0.4), kernels.scaled_sum(kernels.scaled_sum(None, a, 0.75), b, -0.4))
    with pytest.raises(kernels.KernelError):
        kernels.moe_experts_tiled(x, up, down, idx, wt, "relu2", gated=False, opening=extra[:, 0])
    with pytest.raises(kernels.KernelError):
        kernels.scaled_pair(x, 1.0, x.float(), 1.0)


@pytest.mark.parametrize("E,I", [(1, 0), (8, 2), (65, 1), (1024, 0)])
@pytest.mark.parametrize("P,highs", [(1, (0, 64)), (1, (64, 64)), (700, (64, 0)), (900, (64, 64)), (3000, (0, 0)), (5000, (256, 128))])
def test_tiles_of_the_plan(E, I, P, highs):
    """Every expert's slots are covered once, its tiles of one height but the last, no higher than asked for and no more than there can be."""
    from xinfer_amd import kernels
    g = torch.Generator().manual_seed(E + P)
    idx = (torch.rand(P, generator=g) ** 3 * (E + I)).to(torch.int32)
    (h1, m1, c1), (h2, m2, c2) = (kernels._moe_tiles(P, E, h, n, True) for h, n in zip(highs, (3000, 640)))
    order, slot_of = (torch.full((P,), -1, dtype=torch.int32, device=DEV) for _ in range(2))
    lists = [torch.full((5 * m + 3,), -1, dtype=torch.int32, device=DEV) for m in (m1, m2)]
    p, dev = kernels._p, idx.to(DEV)
    kernels._ok(kernels.lib().xi_moe_plan(p(dev), P, E, I, h1, h2, c1, c2, p(order), p(slot_of), p(lists[0]), p(lists[1]), m1, m2, kernels._stream()))
    o, counts = order.cpu().long(), torch.bincount(idx.long(), minlength=E + I).tolist()
    assert sorted(o.tolist()) == list(range(P)) and bool((idx[o][1:] >= idx[o][:-1]).all())
    assert bool((slot_of.cpu().long()[o] == torch.arange(P)).all())
    for tiles, most, high in zip(lists, (m1, m2), highs):
        t = tiles.tolist()
        n, many = t[5 * most], t[5 * most + 1]
        assert 0 <= n <= most and t[5 * most + 2] == -1
        assert highs == (64, 64) or bool(many) == (2 * n > 3 * sum(c > 0 for c in counts[:E])) and many <= 2
        e, row0, rows, first, count = (t[i * most:i * most + n] for i in range(5))
        assert max(rows, default=0) <= (high or 256)
        at = i = 0
        for x in range(E):
            mine = [j for j in range(n) if e[j] == x]
            assert mine == list(range(i, i + len(mine)))
            assert [row0[j] for j in mine] == [at + sum(rows[i:j]) for j in mine] and sum(rows[j] for j in mine) == counts[x]
            assert all(rows[j] == rows[i] for j in mine[:-1]) and all(0 < rows[j] <= rows[i] for j in mine)
            assert all(first[j] == i and count[j] == len(mine) for j in mine)
            at, i = at + counts[x], i + len(mine)


@pytest.mark.parametrize("counts,orders", [([1024] * 8, (2, 2)), ([1000] * 16, (2, 2)), ([700, 130] * 4, (1, 1)), ([128] * 8, (0, 0)),
                                           ([0, 512, 0, 512] * 300, (2, 2)), ([2000] + [60] * 8, (1, 1))])
def test_orders_of_the_tiles(counts, orders):
    """Tiles of about one height go an expert after the other, unequal ones the same columns of all experts to every die, single ones in turn."""
    from xinfer_amd import kernels
    counts = counts[:1024]
    E, P = len(counts), sum(counts)
    dev = torch.repeat_interleave(torch.arange(E), torch.tensor(counts)).to(torch.int32)[torch.randperm(P, generator=torch.Generator().manual_seed(0))].to(DEV)
    (h1, m1, c1), (h2, m2, c2) = (kernels._moe_tiles(P, E, 0, n, False) for n in (6144, 4096))
    order, slot_of = (torch.empty(P, dtype=torch.int32, device=DEV) for _ in range(2))
    lists = [torch.empty(5 * m + 2, dtype=torch.int32, device=DEV) for m in (m1, m2)]
    p = kernels._p
    kernels._ok(kernels.lib().xi_moe_plan(p(dev), P, E, 0, h1, h2, c1, c2, p(order), p(slot_of), p(lists[0]), p(lists[1]), m1, m2, kernels._stream()))
    assert tuple(int(t[5 * m + 1]) for t, m in zip(lists, (m1, m2))) == orders


@pytest.mark.parametrize("E,I", [(1, 0), (63, 2), (64, 0), (65, 1), (1000, 24), (1024, 0)])
@pytest.mark.parametrize("P,bm", [(1, 64), (130, 32), (3000, 64), (5000, 128)])
def test_pairs_in_the_order_of_their_experts(E, I, P, bm):
    """The sort for one expert to the most there are: every pair in one slot, experts in order, tiles as they follow from the counts."""
    from xinfer_amd import kernels
    g = torch.Generator().manual_seed(E + P)
    idx = (torch.rand(P, generator=g) ** 3 * (E + I)).to(torch.int32)             # uneven, some experts without a pair
    most = kernels.lib().xi_moe_tiles_most(P, E, bm)
    order, slot_of = (torch.full((P,), -1, dtype=torch.int32, device=DEV) for _ in range(2))
    lists = [torch.full((most + 1,), -1, dtype=torch.int32, device=DEV) for _ in range(3)]
    n_tiles = torch.zeros(1, dtype=torch.int32, device=DEV)
    dev = idx.to(DEV)
    p = kernels._p
    kernels._ok(kernels.lib().xi_moe_sort(p(dev), P, E, I, bm, p(order), p(slot_of), p(lists[0]), p(lists[1]), p(lists[2]), p(n_tiles), kernels._stream()))
    want, at = [[], [], []], 0
    for e in range(E + I):
        c = int((idx == e).sum())
        for r in range(0, c if e < E else 0, bm):
            for w, v in zip(want, (e, at + r, min(bm, c - r))):
                w.append(v)
        at += c
    n = len(want[0])
    assert n == int(n_tiles) <= most
    for got, w in zip(lists, want):
        assert got[:n].tolist() == w and got[most].item() == -1
    o = order.cpu().long()
    assert sorted(o.tolist()) == list(range(P)) and bool((idx[o][1:] >= idx[o][:-1]).all())
    assert bool((slot_of.cpu().long()[o] == torch.arange(P)).all())


def test_what_is_taken_and_refused():
    from xinfer_amd import kernels
    assert kernels.moe_tiled_takes(100, 2, 8, 128, 192, True)
    assert not kernels.moe_tiled_takes(100, 2, 8, 128, 200, True) and not kernels.moe_tiled_takes(100, 2, 8, 136, 192, True)
    assert not kernels.moe_tiled_takes(1 << 20, 2, 8, 4096, 6144, True)          # rows whose offsets pass 32 bits
    z = lambda *s: torch.zeros(*s, dtype=torch.bfloat16, device=DEV)
    idx = torch.zeros(3, 1, dtype=torch.int32, device=DEV)
    wt = torch.ones(3, 1, device=DEV)
    with pytest.raises(kernels.KernelError):
        kernels.moe_experts_tiled(z(3, 96), z(2, 128, 96), z(2, 96, 64), idx, wt)
    with pytest.raises(kernels.KernelError):
        kernels.moe_experts_tiled(z(3, 64), z(2, 128, 64), z(2, 64, 64), idx, wt, tile_rows=32)


@pytest.mark.parametrize("T", [3, 200])
def test_rows_off_16_bytes(T):
    """Rows may start on any element, as in the other forms."""
    from xinfer_amd import kernels
    g = torch.Generator().manual_seed(T)
    E, H, F = 3, 128, 64
    rb = lambda *s: torch.randn(*s, generator=g).to(torch.bfloat16)
    gate_up, down, x = (rb(E, 2 * F, H) * H ** -0.5).to(DEV), (rb(E, H, F) * F ** -0.5).to(DEV), rb(T, H).to(DEV)
    idx = torch.randint(0, E + 1, (T, 2), generator=g).to(torch.int32).to(DEV)           # (one identity expert)
    wt = torch.rand(T, 2, generator=g).to(DEV)
    flat = torch.zeros(T * H + 1, dtype=torch.bfloat16, device=DEV)
    flat[1:] = x.reshape(-1)
    got = kernels.moe_experts_tiled(flat[1:].view(T, H), gate_up, down, idx, wt, identity=1)
    assert torch.equal(got, kernels.moe_experts_tiled(x, gate_up, down, idx, wt, identity=1))
