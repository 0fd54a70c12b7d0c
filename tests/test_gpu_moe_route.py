"""The router of a mixture of experts over many tokens: every form of its kernel (one, two and four tokens a workgroup; vectors and
single numbers) against float64, and bit for bit beside the same rows in pieces of few tokens."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


# H: less than a round of vectors (single numbers), one round, several, rows that are no whole vectors; T: the edges of the forms and of
# two and four tokens a workgroup
@pytest.mark.parametrize("H", [256, 512, 1000, 1032, 2052])
@pytest.mark.parametrize("T,E,X", [(1, 5, 0), (511, 8, 1), (639, 40, 0), (641, 8, 2), (903, 64, 0), (1023, 10, 1), (1024, 33, 0), (1025, 8, 0), (1027, 64, 3),
                                   (2051, 40, 1), (4098, 9, 1)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_many_tokens(T, E, X, H, dtype):
    from xinfer_amd import kernels
    g = torch.Generator().manual_seed(T + H)
    x = torch.randn(T, H, generator=g).to(dtype)
    w = torch.randn(E + X, H, generator=g) * H ** -0.5
    bias, corr = torch.randn(E, generator=g), torch.rand(E, generator=g) * 0.2
    top = min(4, E)
    xd, wd = x.to(DEV), w.to(DEV)
    z = (xd.double() @ wd.double().t()).cpu()
    # sums of H products of standard deviation 1 / sqrt(H), below 6 in all: H roundings of 2^-24 at worst in one chain
    bound = 6 * (H / 64 + 8) * 2.0 ** -24
    for kind in ("chosen", "all", "sigmoid", "all corrected", "sigmoid corrected"):
        c = corr if "corrected" in kind else None
        kw = dict(all_scores=kind.startswith("all"), sigmoid=kind.startswith("sigmoid"), extra_rows=X, correction=None if c is None else c.to(DEV))
        b = bias if c is None else None
        run = lambda rows: kernels.moe_route(xd[rows], wd, None if b is None else b.to(DEV), top, **kw)
        got = run(slice(0, T))
        for first in range(0, T, 301):
            part = run(slice(first, min(T, first + 301)))
            assert all(torch.equal(p, q[first:first + 301]) for p, q in zip(part, got)), (kind, first)
        idx, wt = got[0].cpu().long(), got[1].cpu().double()
        if X:
            assert float((got[2].cpu().double() - z[:, E:]).abs().max()) < bound
        logit = z[:, :E] + (0.0 if b is None else b.double())
        score = torch.sigmoid(logit) if "sigmoid" in kind else torch.softmax(logit, 1) if "all" in kind else logit
        by = score + c.double() if c is not None else logit
        want = by.topk(top, dim=1).values
        assert float((by.gather(1, idx) - want).abs().max()) < 2 * bound          # (of two that are that close either)
        assert bool((idx.sort(dim=1).values[:, 1:] != idx.sort(dim=1).values[:, :-1]).all())
        s = score.gather(1, idx)
        ref = s if "sigmoid" in kind else torch.softmax(s, 1) if kind == "chosen" else s / (s.sum(1, keepdim=True) + 1e-20)
        # a weight's own error is that of the logits in it, and a few roundings more
        assert float((wt - ref).abs().max()) < 4 * bound + 2.0 ** -21
