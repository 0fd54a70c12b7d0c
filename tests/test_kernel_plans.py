"""What the host decides before a kernel is launched (no GPU): how a narrow product is cut
along K for the many-row tiled kernel, and how a decode step's keys are shared out among workgroups."""
import os
import random
import re
import shutil
import subprocess

import numpy as np
import pytest
import torch

from xinfer_amd import kernels
from xinfer_amd.cache import busiest_over_share
from xinfer_amd.engine.runner import lengths_class

SHAPES = [(6144, 4096), (4096, 4096), (4096, 12288), (7168, 5120), (5120, 5120), (5120, 17408), (10240, 5120),
          (5120, 8192), (5120, 25600), (4096, 1024), (1024, 2048), (1024, 3072), (24576, 4096), (1000, 2056), (48, 96)]


@pytest.mark.parametrize("N,K", SHAPES)
def test_tile_split_plan(N, K):
    """Up to 16 slices of whole tiles of 64 k, the longest slice at least 512 of K, nothing is cut
    up to 128 or beyond 1,024 rows, beyond 256 rows only products with K >= 2 N, and never a weight
    of 8 MB or less."""
    for M in list(range(1, 1300, 7)) + [128, 129, 256, 257, 512, 513, 1024, 1025]:
        s, shape = kernels.tile_split_plan(M, N, K)
        assert 1 <= s <= 16 and shape in (0, 1, 2)
        if s == 1:
            continue
        assert 128 < M <= 1024
        assert K % 64 == 0 and N % 4 == 0
        assert -(-(K // 64) // s) * 64 >= 512 and N * K * 2 > 8 << 20
        assert M <= 256 or K >= 2 * N


def test_tile_split_plan_at_the_sizes_that_were_measured():
    table = {(256, 6144, 4096): (5, 1), (256, 4096, 4096): (6, 1), (256, 4096, 12288): (8, 1), (512, 4096, 12288): (8, 2), (768, 4096, 12288): (5, 2), (1024, 4096, 12288): (4, 2), (512, 4096, 4096): (1, 0), (512, 6144, 4096): (1, 0), (256, 7168, 5120): (4, 1), (256, 5120, 5120): (5, 1), (256, 5120, 17408): (6, 1), (256, 1024, 2048): (1, 0), (256, 1024, 3072): (1, 0), (192, 4096, 12288): (8, 1), (129, 4096, 4096): (8, 1), (200, 1000, 2056): (1, 0), (256, 5120, 25600): (6, 1), (512, 5120, 17408): (6, 2), (256, 10240, 5120): (3, 1)}
    for (M, N, K), want in table.items():
        assert kernels.tile_split_plan(M, N, K) == want, (M, N, K)


@pytest.mark.parametrize("similar", [False, True])
def test_decode_keys_per_workgroup_is_a_multiple_of_128_and_covers_the_span(similar):
    for pairs in (1, 8, 64, 96, 256, 512, 2048):
        for span in (1, 100, 1024, 4096, 8704, 32768, 131072):
            kpw = kernels.decode_keys_per_workgroup(pairs, span, similar)
            assert kpw >= 128 and kpw % 128 == 0
            assert span // kpw + 1 <= 1025


def test_decode_mixed_lengths_take_whole_sequences_where_there_are_many():
    assert kernels.decode_keys_per_workgroup(255, 4096, False) == 512
    assert kernels.decode_keys_per_workgroup(256, 4096, False) == 1024             # a pair a compute unit
    assert kernels.decode_keys_per_workgroup(256, 1024, False) == 512
    assert kernels.decode_keys_per_workgroup(383, 1024, False) == 512
    assert kernels.decode_keys_per_workgroup(384, 1024, False) == 1152             # one split: no second kernel
    assert kernels.decode_keys_per_workgroup(1536, 2048, False) == 2176
    assert kernels.decode_keys_per_workgroup(2048, 3072, False) == 2048
    assert kernels.decode_keys_per_workgroup(2048, 16384, False) == 2048


def test_decode_keys_per_workgroup_of_even_lengths():
    plan = lambda pairs, span: kernels.decode_keys_per_workgroup(pairs, span, kernels.EVEN_LENGTHS)
    assert plan(488, 3072) == 3200 and plan(264, 2048) == 2176 and plan(240, 1024) == 1152 and plan(4096, 4096) == 4224
    for pairs, span in ((217, 1024), (184, 2048), (256, 4096), (8, 1024), (600, 5000)):
        assert plan(pairs, span) == kernels.decode_keys_per_workgroup(pairs, span, False)



def test_float32_attention_sets_one_limit_a_kernel():
    """The dynamic LDS that the kernel of a class of head sizes is allowed: one number for the class, enough for all of it, so that
    two engines with different heads do not lower it between each other's setting and launch."""
    limit = kernels.lib().xi_attention_f32_lds
    sizes = [(d, dv) for d in range(16, 257, 16) for dv in range(16, 257, 16)]
    kinds = {}
    for d, dv in sizes:
        kinds.setdefault(next(m for m in (64, 128, 256) if max(d, dv) <= m), set()).add(limit(d, dv))
        need = 4 * (8 * (16 * dv + 32) + 16 * (d + 4))          # eight waves' sums of 16 rows, their maxima and totals, the queries
        assert need <= limit(d, dv) <= 160 * 1024
    assert all(len(v) == 1 for v in kinds.values())


@pytest.mark.parametrize("lens,H,dk,dv,walk", [
    ([2048], 1, 128, 64, False), ([2304], 1, 128, 64, False), ([3072], 1, 128, 64, True), ([8192], 8, 128, 64, True),
    ([4096], 8, 128, 64, True), ([8192], 16, 128, 64, False), ([8192], 128, 128, 64, False), ([3000, 3000], 8, 128, 64, False),
    ([8192], 1, 32, 32, True), ([2816], 1, 32, 32, False), ([4096, 64, 300], 8, 128, 64, False), ([1] * 60, 8, 64, 64, False)])
def test_few_heads_walk_a_long_portion_side_by_side(lens, H, dk, dv, walk, monkeypatch):
    import torch
    assert kernels.step_walk_ahead(lens, H, dk, dv) == walk
    # the route that `linear_scan` takes, without a launch
    taken = []
    monkeypatch.setattr(kernels, "_stream", lambda: 0)
    monkeypatch.setattr(kernels, "_ok", lambda rc: None)

    class Lib:
        xi_step_chunks_takes = staticmethod(lambda dk, dv: 1)

        def __getattr__(self, name):
            return lambda *a: taken.append(name)

    monkeypatch.setattr(kernels, "lib", lambda: Lib())
    T = sum(lens)
    t = torch.empty(1, dtype=torch.bfloat16)
    common = (t, t, t, 8, 8, 8, None, None, 1.0, None, t, H, t, t, None, dv, H, 0)
    cu_q = torch.zeros(len(lens) + 1, dtype=torch.int32)
    done = kernels._step_chunks(common, t, H * dk * dv, torch.arange(len(lens)), cu_q, lens, {}, t, H, dk, dv, 1.0, 1.0)
    assert done == (not walk and max(lens) >= kernels.STEP_FROM)
    assert taken[:1] == (["xi_step_chunks"] if done else [])


@pytest.mark.parametrize("bm", [32, 64, 128, 256])
def test_most_tiles_of_routed_experts(bm):
    """The largest number of tiles that any sharing out of the pairs makes, and no more."""
    most = kernels.lib().xi_moe_tiles_most
    for P in (1, 2, 7, 31, 32, 33, 64, 65, 200, 257, 1000, 4097):
        for E in (1, 2, 3, 8, 100, 1024):
            # one pair for every expert that gets any, bm more for as many tiles as the rest gives, the remainder anywhere
            n = min(P, E)
            counts = [1] * n
            full, rest = divmod(P - n, bm)
            for i in range(full):
                counts[i % n] += bm
            assert sum(-(-c // bm) for c in counts) == most(P, E, bm)
            counts[0] += rest
            assert sum(-(-c // bm) for c in counts) == most(P, E, bm)
            even = [P // n + (i < P % n) for i in range(n)]
            assert sum(-(-c // bm) for c in even) <= most(P, E, bm)
            assert -(-P // bm) <= most(P, E, bm)


def test_float32_attention_tiles():
    """Tokens a workgroup: the fewest that make one round of workgroups, at most 16 (token, head) rows, one for single tokens."""
    from xinfer_amd import kernels
    tile = kernels.lib().xi_attention_f32_tile
    assert [tile(n, 1, 16, 16) for n in (1, 16, 17, 20, 64, 128, 240, 256, 257, 2048)] == [1, 1, 2, 2, 4, 8, 15, 16, 16, 16]
    assert [tile(n, 1, 32, 8) for n in (20, 32, 33, 64, 2048)] == [1, 1, 2, 2, 4]
    assert tile(2048, 1, 40, 1) == 1 and tile(4000, 1, 12, 4) == 5
    assert tile(64, 64, 16, 16) == 1 and tile(64, 17, 16, 16) == 1 and tile(64, 16, 16, 16) == 4


def test_leading_singles():
    from types import SimpleNamespace
    import torch
    from xinfer_amd import kernels
    f, b = torch.zeros(1), torch.zeros(1, dtype=torch.bfloat16)
    ctx = lambda cu, most: SimpleNamespace(cu_q_host=cu, max_q_len=most, scratch={})
    assert kernels.leading_singles(f, ctx([0, 1, 2, 9, 10], 7)) == 2
    assert kernels.leading_singles(f, ctx([0, 7, 8], 7)) == 0
    assert kernels.leading_singles(f, ctx((), 1)) == 0 and kernels.leading_singles(b, ctx([0, 1, 9], 8)) == 0


def test_float32_product_forms():
    """Tiles for short K and narrow outputs of many rows, the kernel for few rows, and the cut tiles, by size; every launch within 2^32 threads."""
    from xinfer_amd import kernels
    form = kernels.gemm_f32_form
    assert form(1 << 20, 16, 128) == 5 and form(1 << 29, 16, 4096) == 5 and form(2048, 1024, 16) == 5
    assert form(8, 4096, 4096) == 0 and form(8, 24576, 4096) == 1 and form(4096, 16, 4096) == 0
    assert form(200, 4096, 4096) == 2 and form(562, 151936, 4096) == 3 and form(562, 4096, 4096) == 4
    assert form(40000, 4096, 256) == 5 and form(2048, 4096, 256) == 4         # 2,048 rows at a time leave gaps
    assert form(8, 151936, 4096) == 1 and form(32, 24576, 4096) == 1          # wide outputs of few rows: bound by the weights
    # ... at K = 1024 too, where a workgroup's start counts once and not for every tile it walks; and weights from memory behind tiles for short K
    assert form(1, 151936, 1024) == 0 and form(8, 151936, 1024) == 1 and form(100, 6144, 1024) == 1 and form(600, 1024, 3072) == 1
    scratch = lambda M, N, K: int(kernels.lib().xi_gemm_f32_scratch(M, N, K, -1))
    assert scratch(1 << 20, 16, 128) == 0 and scratch(562, 4096, 4096) == 6 * 4096 * 562 and scratch(100_000, 4096, 4096) == 6 * 4096 * 2048


def test_three_parts_of_a_float32():
    """2^24 of any float32 up to 2^104 is the sum of three bfloat16, none of them subnormal, and what the six products of two numbers leave out is at most
    2^-24 + 2^-34 of theirs."""
    import torch
    g = torch.Generator().manual_seed(0)
    worst = torch.tensor([float.fromhex(h) for h in ("0x1.00ff8p+0", "0x1.01p+0", "0x1.fffffep+0", "0x1.00fffep+0", "0x1p-149", "0x1.fffffep-127", "0x1.fcp+103")])
    x = torch.cat([worst, -worst, torch.randn(1 << 20, generator=g), torch.randn(1 << 20, generator=g) * 2.0 ** -110 * 2.0 ** -16])

    def parts(x):
        rest, out = x * 2.0 ** 24, []
        for _ in range(3):
            out.append(rest.to(torch.bfloat16))
            rest = rest - out[-1].float()
        assert bool((rest == 0).all())
        return [p.double() for p in out]

    hi, mid, lo = parts(x)
    assert torch.equal(hi + mid + lo, x.double() * 2.0 ** 24)
    assert all(bool(((p == 0) | (p.abs() >= 2.0 ** -126)).all()) for p in (hi, mid, lo))
    perm = torch.cat([torch.arange(len(worst)), len(worst) + torch.randperm(len(x) - len(worst), generator=g)])
    out = mid * lo[perm] + lo * mid[perm] + lo * lo[perm]
    assert bool((out.abs() <= (2.0 ** -24 + 2.0 ** -34) * (x.double() * x.double()[perm]).abs() * 2.0 ** 48).all())


def test_round_tiles_ahead():
    """One full round of tiles of 256 by 128, long K."""
    ahead = kernels.round_tiles_ahead
    assert ahead(2048, 4096, 12288) and ahead(1793, 4096, 6144) and ahead(1537 - 256, 5120, 5120) and ahead(1025, 6144, 20480)
    assert ahead(1792, 4096, 8192) and not ahead(1791 - 255, 4096, 8192)       # 7 x 32 tiles, 6 x 32
    for M, N, K in ((2048, 4096, 4096), (2049, 4096, 12288), (1536, 4096, 12288), (2048, 2048, 8192), (4096, 2048, 16384), (8, 4096, 12288)):
        assert not ahead(M, N, K), (M, N, K)


def test_loads_into_lds_wait_for_m0():
    """An asm that writes m0 and loads into LDS behind it has the wait state that the pair wants: the compiler puts none inside an asm."""
    folder = os.path.join(os.path.dirname(kernels.__file__), "csrc", "kernels")
    found = 0
    for name in sorted(os.listdir(folder)):
        with open(os.path.join(folder, name)) as f:
            for text in re.findall(r'asm volatile\("((?:[^"\\]|\\.)*)"', f.read()):
                lines = [line.strip() for line in text.replace("\\t", "").split("\\n")]
                for before, line in zip(lines, lines[1:] + [""]):
                    if re.match(r"s_\w+ m0,", before):
                        found += 1
                        assert line.startswith("s_nop"), (name, text)
    assert found >= 4


def test_a_steps_small_array_is_not_recorded(monkeypatch):
    """While a graph is recorded the copy from a pinned block, which is another array's by the next replay, is refused as one from ordinary
    memory is; on the CPU it is a plain tensor."""
    assert kernels.on_device([[1, 2], [3, 4]], torch.int32, "cpu").tolist() == [[1, 2], [3, 4]]
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: True)
    made = []
    monkeypatch.setattr(torch, "empty", lambda *a, **kw: made.append(kw))
    with pytest.raises(kernels.KernelError, match="recorded"):
        kernels.on_device([1, 2], torch.int64, "cuda:0")
    assert not made


def test_even_lengths_are_read_by_the_kernel_they_were_measured_in(monkeypatch):
    """A step of even lengths goes as whole sequences in the kernel for whole-rotated heads without bias or window on pages of 32 keys and
    more; with q given, a bias, a window, small pages, half of a head turned or pairs (2i, 2i + 1) it is cut up as lengths of any kind are."""
    real, cut = kernels.lib(), []

    class Noted:
        def __getattr__(self, name):
            if not name.startswith("xi_attention_decode_") or name == "xi_attention_decode_lean":
                return getattr(real, name)
            return lambda *args: cut.append(int(args[-9])) or 0
    monkeypatch.setattr(kernels, "lib", Noted)
    monkeypatch.setattr(kernels, "_dev", lambda *a: None)
    monkeypatch.setattr(kernels, "_stream", lambda: None)
    bf = lambda *shape: torch.zeros(shape, dtype=torch.bfloat16)
    i32 = lambda *shape: torch.zeros(shape, dtype=torch.int32)
    B, nq, nkv, d, span = 264, 2, 1, 64, 2048

    def packed(page=64, rot=d, interleaved=False, bias=None, window=0, slices=0, similar=kernels.EVEN_LENGTHS):
        cut.clear()
        qkv = torch.zeros(slices, B, (nq + 2 * nkv) * d) if slices else bf(B, (nq + 2 * nkv) * d)
        kernels.attention_decode_packed_bf16(qkv, None, None, 1e-6, torch.zeros(4, rot // 2), torch.zeros(4, rot // 2), rot, interleaved, i32(B),
                                             torch.zeros(B, dtype=torch.int64), bf(1, nkv, page, d), bf(1, nkv, page // 8, d, 8), i32(B, 1), i32(B), span, nq,
                                             0.1, window, bias=bias, similar=similar)
        return cut[0]
    whole, mixed = 2176, kernels.decode_keys_per_workgroup(B * nkv, span, False)
    assert whole != mixed
    assert packed() == packed(slices=8) == whole and packed(similar=False) == mixed
    for other in (dict(page=16), dict(rot=32), dict(interleaved=True), dict(bias=torch.zeros((nq + 2 * nkv) * d)), dict(slices=9)):
        assert packed(**other) == mixed, other
    assert packed(window=span) == packed(window=span, similar=False)
    for similar in (kernels.EVEN_LENGTHS, False):
        cut.clear()
        kernels.attention_decode_bf16(bf(B, nq, d), bf(1, nkv, 64, d), bf(1, nkv, 8, d, 8), i32(B, 1), i32(B), span, 0.1, similar=similar)
        assert cut == [mixed]


def _dealt_out(lengths, columns):
    """Longest first, each to the column with the fewest keys: the busiest one's keys beyond the share, rounded down."""
    keys = [0] * columns
    for n in sorted(lengths, reverse=True):
        keys[keys.index(min(keys))] += n
    return max(keys) - sum(keys) // columns


def test_busiest_over_share():
    rng = random.Random(5)
    for n, columns in ((1, 1), (3, 32), (16, 32), (33, 32), (61, 32), (200, 85), (256, 8), (17, 1)):
        lengths = [rng.randint(1, 1 << rng.randint(0, 20)) for _ in range(n)]
        assert busiest_over_share(np.asarray(lengths, np.int32), columns) == _dealt_out(lengths, columns), (n, columns)
    assert busiest_over_share(np.empty(0, np.int32), 32) == 0
    most = [2 ** 31 - 1] * 40                       # (sums beyond an int; the excess itself is never more than the longest)
    assert busiest_over_share(np.asarray(most, np.int32), 39) == _dealt_out(most, 39)


def test_lengths_class_looks_at_how_the_sequences_deal_out():
    """Not the mean alone: one full round of long sequences and a few more leave most of the chip idle, whatever the short ones beside them."""
    of = lambda lengths, heads=(8,), **kw: lengths_class(np.asarray(lengths, np.int32), 1 + max(lengths, default=0), heads, **kw)
    rng = random.Random(6)
    ragged = [rng.randint(90, 2700) for _ in range(61)]
    assert of(ragged) == kernels.EVEN_LENGTHS and of(sorted(ragged)) == kernels.EVEN_LENGTHS
    for n, longest, short in ((33, 4000, 15), (38, 4000, 10), (39, 3300, 61), (36, 4000, 54), (35, 2700, 37), (16, 4000, 24), (11, 2700, 17)):
        assert of([longest] * n + [100] * short) is False, (n, longest, short)
    assert of([4000] * 8) is True and of([3900] * 30 + [4000] * 30) is True and of([900] * 30, similar=False) == kernels.EVEN_LENGTHS
    assert of(ragged[:15]) is False and of(ragged, ()) is False and of([]) is False
    # several numbers of kv heads: every one has to deal out
    uneven = [1800] * 33 + [100] * 12
    assert of(uneven, (8,)) is False and of(uneven, (16,)) is False and of(uneven, (6,)) == kernels.EVEN_LENGTHS and of(uneven, (6, 8)) is False


def test_lengths_class_is_told_only_where_a_plan_differs():
    """The class is part of a recorded step's key: lengths that drift over the line do not record the same kernels again."""
    of = lambda lengths, span, heads: lengths_class(np.asarray(lengths, np.int32), span, heads)
    told = 0
    for B in (16, 20, 27, 28, 32, 48, 61, 64, 200, 256):
        ragged = [20 + 5 * i for i in range(B)]
        assert not of(ragged, 8192, ()) and of([500] * B, 1024, ()) is True
        for span in range(1024, 9 * 1024, 1024):
            got = of(ragged, span, (8,))
            assert got in (False, kernels.EVEN_LENGTHS)
            told += bool(got)
            differs = kernels.decode_keys_per_workgroup(8 * B, span, kernels.EVEN_LENGTHS) != kernels.decode_keys_per_workgroup(8 * B, span, False)
            assert bool(got) == differs, (B, span)        # (these lengths deal out)
            if B < 28 or span > 4096 or (B >= 48 and span <= 2048):
                assert not got, (B, span)
    assert told


def test_moe_tiles_of_few_rows_where_no_expert_has_many():
    """Steps of up to 16 tokens have at most 16 rows an expert, however they share out; longer ones may put most pairs on a few experts."""
    rows = lambda T, top, E: kernels.moe_tile_rows(T * top, E, 768, 1024, True, T)
    assert rows(8, 2, 8) == rows(16, 4, 8) == rows(1, 8, 1000) == rows(17, 2, 16) == rows(64, 4, 64) == rows(16, 8, 16) == (16, 16)
    assert rows(16, 5, 8) == rows(17, 2, 8) == rows(32, 2, 8) == rows(65, 4, 64) == rows(128, 8, 128) == rows(64, 8, 64) == (64, 64)


def test_thin_products_ask_for_all_of_k_where_it_was_ahead():
    """Tiles of 512 k that few-row products ask for together: up to 1,024 of K with any rows, 2,048 with up to 8 and 1,536 with more; workgroups of
    up to four features that add into the stream 2,048, and 3,072 with up to 8 rows.  Longer K, 0, is walked; -1: no such tiles."""
    depth = kernels.lib().xi_linear_thin_depth
    for N, adds, most in ((1024, 0, {8: 2048, 16: 1536}), (2048, 0, {8: 2048, 16: 1536}), (2048, 1, {8: 2048, 16: 1536}), (1024, 1, {8: 3072, 16: 2048}),
                          (256, 1, {8: 3072, 16: 2048}), (4096, 1, {8: 2048, 16: 1536})):
        for M in (1, 4, 8, 9, 16):
            for K in range(512, 8192, 512):
                got = depth(M, N, K, adds)
                assert (got > 0) == (K <= most[8 if M <= 8 else 16]) and (got == 0 or 512 * got >= K), (N, adds, M, K, got)
    assert depth(1, 8192, 1024, 0) == -1 and depth(1, 1024, 768, 0) == -1 and depth(1, 1024, 100, 0) == -1


def test_round_tiles_of_few_features_leave_strides_of_powers_of_two_alone():
    ahead = kernels.round_tiles_ahead
    for M, N in ((3584, 2048), (4096, 2048), (4352, 1920), (3072, 2560)):
        for K in (5120, 6144, 7168, 10240, 12288, 14336, 17408, 20480):
            assert ahead(M, N, K), (M, N, K)
        for K in (4096, 7232, 8192, 8256, 9216, 14400, 15360, 16320, 16384, 16448, 17344, 20544, 24576, 32768):
            assert not ahead(M, N, K), (M, N, K)
    for K in (5120, 8192, 15360, 16384, 24576):
        assert ahead(2048, 4096, K) and ahead(2560, 3072, K)
    assert not ahead(2048, 4096, 24640) and not ahead(2048, 4096, 32768) and not ahead(2048, 4096, 4096)


@pytest.mark.skipif(shutil.which("hipcc") is None, reason="needs the compiler")
@pytest.mark.parametrize("name", ["linear_thin", "linear_mid"])
def test_folded_products_wait_for_their_parts(name, tmp_path):
    """In the compiled kernels the loads that bring the rows' parts into LDS are issued before the first operands, and the count that is
    waited for behind them is not more than what has been issued since: it waits for the parts."""
    from xinfer_amd.csrc import build
    out = tmp_path / "k.s"
    subprocess.run(["hipcc", *build.HIP_FLAGS, "--offload-device-only", "-S", os.path.join(build.KERNEL_DIR, name + ".hip"), "-o", str(out)], check=True,
                   capture_output=True, timeout=300)
    found = 0
    for kernel, body in re.findall(r"^(_ZN2xi\w+):(.*?)s_endpgm", out.read_text(), re.S | re.M):
        lines = [line.strip() for line in body.split("\n")]
        parts = [i for i, line in enumerate(lines) if line.startswith("global_load_lds_dword ")]
        if not parts:
            continue
        found += 1
        loads = [i for i, line in enumerate(lines) if line.startswith("global_load_dwordx4 ")]
        wait = next(i for i, line in enumerate(lines) if i > parts[-1] and line.startswith("s_waitcnt vmcnt("))
        count = int(re.search(r"vmcnt\((\d+)\)", lines[wait])[1])
        assert min(loads) > parts[-1] and count <= sum(parts[-1] < i < wait for i in loads), kernel
    assert found
