"""A selective state space's long portions on the matrix cores (`xi_step_chunks`) against float64 and beside the walk token by
token: unequal requests, portions at the edges of a chunk of 64 tokens, columns of a packed projection, slots in no order,
decays from none to all within a token."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _plain(q, k, v, raw, bias, rate_log, S, group_heads, q_scale, k_scale):
    """One portion in float64; returns the results and the state behind it."""
    H, T = raw.shape[1], q.shape[0]
    dk = S.shape[1]
    q, k = ((t.double().view(T, -1, dk) * s).repeat_interleave(group_heads, dim=1) for t, s in ((q, q_scale), (k, k_scale)))
    v = v.double().view(T, H, -1)
    x = raw.double() + bias.double()
    d = torch.logaddexp(x, torch.zeros_like(x))
    a = torch.exp(-torch.exp(rate_log.double()) * d)
    S = S.double().clone()
    out = []
    for t in range(T):
        S = a[t][:, None, None] * S + k[t][:, :, None] * (d[t][:, None] * v[t])[:, None, :]
        out.append((S * q[t][:, :, None]).sum(1))
    return torch.stack(out), S


@pytest.mark.parametrize("H,G,dk,dv,rate", [(4, 1, 128, 64, -1.0), (6, 2, 32, 32, -6.0), (2, 2, 96, 96, 3.0), (3, 1, 64, 32, 0.5)])
def test_portions_of_unequal_requests(H, G, dk, dv, rate, monkeypatch):
    from xinfer_amd import kernels
    g = torch.Generator().manual_seed(dk + dv)
    steps = [[64, 1, 32, 200], [65, 31, 129, 1], [1, 63, 33, 128]]
    B, slots = 4, [2, 0, 4, 3]
    bias, rate_log = torch.randn(H, generator=g) - 1.0, torch.randn(H, generator=g) * 0.5 + rate
    state0 = torch.randn(5, H, dk, dv, generator=g)
    errors = {}
    for matrix in (False, True):
        monkeypatch.setattr(kernels, "STEP_MFMA", matrix)
        g2 = torch.Generator().manual_seed(5)
        state = state0.clone().to(DEV)
        want = {b: state0[s] for b, s in enumerate(slots)}
        worst = [0.0, 0.0]
        for lens in steps:
            T = sum(lens)
            width = 2 * G * dk + H * dv
            packed = torch.randn(T, width + 8 + H, generator=g2).to(torch.bfloat16)
            dev = packed.to(DEV)
            cols = lambda t: (t[:, :G * dk], t[:, G * dk:2 * G * dk], t[:, 2 * G * dk:width], t[:, width + 8:width + 8 + H])
            if (width + 8 + H) % 8:          # rows of whole 16-byte pieces for q, k and v; the step sizes lie anywhere
                pad = torch.zeros(T, -(width + 8 + H) % 8, dtype=torch.bfloat16)
                dev = torch.cat([packed, pad], dim=1).to(DEV)
            q, k, v, raw = cols(dev)
            cu = [0]
            for n in lens:
                cu.append(cu[-1] + n)
            o = kernels.linear_scan(q, k, v, state, torch.tensor(slots, device=DEV), torch.tensor(cu, dtype=torch.int32, device=DEV), H, dk,
                                    dv, step=raw, step_bias=bias.to(DEV), decay_log=rate_log.to(DEV), groups=G, q_scale=0.7, k_scale=0.4,
                                    q_lens=lens, plan_cache={})
            for b in range(B):
                part = [c[cu[b]:cu[b + 1]] for c in cols(packed)]
                ref, want[b] = _plain(*part[:3], part[3], bias, rate_log, want[b], H // G, 0.7, 0.4)
                worst[0] = max(worst[0], float((o[cu[b]:cu[b + 1]].cpu().double() - ref).norm() / ref.norm()))
                worst[1] = max(worst[1], float((state[slots[b]].cpu().double() - want[b]).norm() / want[b].norm()))
        untouched = [s for s in range(5) if s not in slots]
        assert torch.equal(state[untouched].cpu(), state0[untouched])
        errors[matrix] = worst
    print(f"\n[step_chunks] dk={dk} dv={dv}: error of results and state against 64 bits: walk {errors[False]}, chunks {errors[True]}")
    # three bfloat16 hold a float32 to 2^-24 of it, and both forms round float32 sums of at most 64 + dk terms
    for w, c in zip(errors[False], errors[True]):
        assert c < max(1.2 * w, 5e-7)


def _portion(seed, T, H, dk, dv, device=DEV):
    """One request's operands (one group) as `_plain` takes them, and as `linear_scan` does."""
    g = torch.Generator().manual_seed(seed)
    rb = lambda *s: torch.randn(*s, generator=g).to(torch.bfloat16)
    q, k, v, raw = rb(T, dk), rb(T, dk), rb(T, H * dv), rb(T, H)
    bias, rate_log = torch.randn(H, generator=g) - 1.0, torch.randn(H, generator=g) * 0.5 - 1.0
    return q, k, v, raw, bias, rate_log, torch.randn(1, H, dk, dv, generator=g)


def _walk(monkeypatch, matrix, q, k, v, raw, bias, rate_log, state):
    from xinfer_amd import kernels
    monkeypatch.setattr(kernels, "STEP_MFMA", matrix)
    T, (_, H, dk, dv) = q.shape[0], state.shape
    st = state.to(DEV)
    o = kernels.linear_scan(q.to(DEV), k.to(DEV), v.to(DEV), st, torch.zeros(1, dtype=torch.int64, device=DEV),
                            torch.tensor([0, T], dtype=torch.int32, device=DEV), H, dk, dv, step=raw.to(DEV), step_bias=bias.to(DEV),
                            decay_log=rate_log.to(DEV), groups=1, q_lens=[T])
    return o.cpu(), st[0].cpu()


@pytest.mark.parametrize("at", [0, 41, 63, 64])
@pytest.mark.parametrize("size", [3e4, 1e9, 1e20])
def test_a_token_that_forgets_everything(at, size, monkeypatch):
    """A step size that leaves nothing of the state: the decays of the tokens behind it keep their digits."""
    x = _portion(int(size) % 1000 + at, 150, 3, 64, 64)
    x[3][at, 1] = size
    ref, state = _plain(*x[:6], x[6][0], 3, 1.0, 1.0)
    size, state_size = _plain(x[0].abs(), x[1].abs(), x[2].abs(), *x[3:6], x[6][0].abs(), 3, 1.0, 1.0)       # of the terms, all added up
    # dk + 64 roundings of sums of the terms, and the decays' exponents in float32, up to 2^5 where what they scale still counts
    bound = (64 + 64 + 32) * 2.0 ** -24
    for matrix in (False, True):
        o, st = _walk(monkeypatch, matrix, *x)
        assert float(((o.double() - ref).abs() / size).max()) < bound, matrix
        assert float(((st.double() - state).abs() / state_size).max()) < bound, matrix


INF, NAN = float("inf"), float("nan")


@pytest.mark.parametrize("what,values", [("v", (INF, NAN, 1e34, -1e30)), ("k", (INF, NAN, 1e34)), ("q", (-INF, NAN, 1e36)),
                                         ("raw", (INF, NAN, 1e34, -INF)), ("state", (INF, NAN, 3.395e38))])
@pytest.mark.parametrize("dk,dv,at", [(64, 64, 41), (128, 32, 64), (32, 32, 127), (96, 32, 0)])
def test_values_without_a_bound(what, values, dk, dv, at, monkeypatch):
    """An infinite, undefined or very large value in the operands: the same results are finite, infinite and undefined as where the
    walk goes token by token, none of them in front of the value, and the finite ones agree."""
    T, H = 150, 2
    for value in values:
        x = _portion(at + dk, T, H, dk, dv)
        if what == "state":
            x[6][0, 1, 3, 5] = value
        else:
            x[("q", "k", "v", "raw").index(what)][at, 1] = value
        (wo, ws), (co, cs) = _walk(monkeypatch, False, *x), _walk(monkeypatch, True, *x)
        before = 0 if what == "state" else at
        assert bool(co[:before].isfinite().all()), value
        for w, c in ((wo, co), (ws, cs)):
            assert torch.equal(w.isnan(), c.isnan()) and torch.equal(w.isinf(), c.isinf()), value
            assert torch.equal(w[w.isinf()], c[w.isinf()]), value
            fine = w.isfinite()
            # two float32 sums of dk + 64 terms in different orders; a sum in front of which a large term has decayed again
            # keeps that term's rounding, so the error is taken against the largest of the column's finite values
            most = torch.where(fine, w, 0.0).abs().amax(dim=0, keepdim=True)
            assert float(torch.where(fine, (w - c).abs() / most.clamp(min=1.0), torch.zeros(())).max()) < (dk + 64) * 2.0 ** -23, value


def test_short_portions_bring_no_plan_to_the_device(monkeypatch):
    """A step whose portions are all walked token by token copies nothing for the chunks' sake."""
    from xinfer_amd import kernels
    x = _portion(1, 40, 2, 32, 32)
    q, k, v, raw, bias, rate_log, state = (t.to(DEV) for t in x)
    kept = {}
    st = state.expand(3, -1, -1, -1).contiguous()
    kernels.linear_scan(q, k, v, st, torch.arange(3, device=DEV), torch.tensor([0, 31, 32, 40], dtype=torch.int32, device=DEV), 2, 32, 32,
                        step=raw, step_bias=bias, decay_log=rate_log, groups=1, q_lens=[31, 1, 8], plan_cache=kept)
    assert not [k for plan in kept.values() for k, t in plan.items() if torch.is_tensor(t)]


def test_steps_of_both_kinds_make_no_arrays():
    """Rows of either kind between those of the other are passed over: the bits of each portion by itself, and nothing copied for it."""
    from xinfer_amd import kernels
    H, dk, dv = 2, 64, 32
    for lens in ([40], [64, 90], [1, 1, 40, 70], [70, 3, 1], [5, 33, 1, 64, 31, 200, 2], [64, 1, 64]):
        x = _portion(len(lens), sum(lens), H, dk, dv)
        q, k, v, raw, bias, rate_log, state = (t.to(DEV) for t in x)
        B = len(lens)
        slots = torch.arange(B, device=DEV).flip(0)
        cu = [sum(lens[:i]) for i in range(B + 1)]
        run = lambda st, sl, a, b, n, kept: kernels.linear_scan(
            q[a:b], k[a:b], v[a:b], st, sl, torch.tensor([sum(n[:i]) for i in range(len(n) + 1)], dtype=torch.int32, device=DEV), H, dk, dv,
            step=raw[a:b], step_bias=bias, decay_log=rate_log, groups=1, q_lens=n, plan_cache=kept)
        both, single, kept = state.repeat(B, 1, 1, 1), state.repeat(B, 1, 1, 1), {}
        got = run(both, slots, 0, cu[B], lens, kept)
        for i in range(B):
            assert torch.equal(got[cu[i]:cu[i + 1]], run(single, slots[i:i + 1].contiguous(), cu[i], cu[i + 1], lens[i:i + 1], {})), (lens, i)
        assert torch.equal(both, single), lens
        assert not [k for plan in kept.values() for k, t in plan.items() if torch.is_tensor(t)]


def test_the_rule_takes_what_it_should(monkeypatch):
    """Which portions go where, without a launch."""
    from xinfer_amd import kernels
    assert kernels.step_chunk_plan([1, 31, 32, 500, 1]) == ([0, 1, 4], [2, 3])
    takes = kernels.lib().xi_step_chunks_takes
    assert all(takes(dk, dv) for dk in (32, 64, 96, 128) for dv in (32, 64, 256))
    assert not any(takes(*s) for s in ((16, 64), (160, 64), (48, 64), (128, 48), (128, 0), (0, 64)))
