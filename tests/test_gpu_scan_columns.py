"""The chunked walk of a decaying state with two value columns a lane: the same bits as the columns' own walks."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("H,dk,dv,dtype", [(8, 128, 256, torch.bfloat16), (9, 100, 200, torch.float32), (32, 20, 65, torch.bfloat16)])
def test_two_columns_a_lane(H, dk, dv, dtype):
    from xinfer_amd import kernels
    g = torch.Generator().manual_seed(dk)
    lens = [1201, 3, 850]
    T = sum(lens)
    cu = torch.tensor([0, 1201, 1204, T], dtype=torch.int32, device=DEV)
    slots = torch.tensor([2, 0, 1], device=DEV)
    q, k = (torch.randn(T, H * dk, generator=g).to(dtype).to(DEV) for _ in range(2))
    v = torch.randn(T, H, dv, generator=g).to(dtype).to(DEV)
    z, zb = torch.randn(T, H * dk, generator=g).to(DEV), torch.randn(H * dk, generator=g).to(DEV)
    state = torch.randn(3, H, dk, dv, generator=g).to(DEV)

    def walk(a, b):
        st = state[..., a:b].clone(memory_format=torch.contiguous_format)
        o = kernels.linear_scan(q, k, v[..., a:b].reshape(T, -1).contiguous(), st, slots, cu, H, dk, b - a, z=z, z_bias=zb, tau=16.0,
                                q_scale=dk ** -0.5, q_lens=lens)
        return o.view(T, H, b - a), st

    whole, st = walk(0, dv)
    for a in range(0, dv, 64):
        part, own = walk(a, min(dv, a + 64))       # up to 64 columns: one a lane
        assert torch.equal(whole[..., a:a + 64], part) and torch.equal(st[..., a:a + 64], own)


def _plain(q, k, v, decay, weight, S, q_scale):
    """One request in float64, from the state S [H, dk, dv]: decay, weight [T, H]; v [T, H, dv]."""
    S, out = S.double().clone(), []
    for t in range(q.shape[0]):
        S = decay[t][:, None, None] * S + k[t][:, :, None] * (weight[t][:, None] * v[t])[:, None, :]
        out.append((S * (q[t] * q_scale)[:, :, None]).sum(1))
    return torch.stack(out), S


@pytest.mark.parametrize("how,dtype", [("gates", torch.bfloat16), ("gates", torch.float32), ("silu", torch.float32), ("step", torch.float32)])
@pytest.mark.parametrize("H,dk,vc", [(16, 64, 129), (11, 100, 200)])
def test_other_decays_with_two_columns_a_lane(how, dtype, H, dk, vc):
    """Ready-made gates beside the keys' own sum (a state's last column), one decay a head under silu, and a step size: enough chunks
    that a lane has two columns, against float64 and against walks of up to 64 columns."""
    from xinfer_amd import kernels
    g = torch.Generator().manual_seed(dk + vc)
    lens = [1130, 2, 901]
    T = sum(lens)
    cu = torch.tensor([0, 1130, 1132, T], dtype=torch.int32, device=DEV)
    chunks = len(kernels.scan_chunk_plan(lens)[2])
    assert chunks * H * -(-vc // 128) >= 512           # xi_linear_scan's rule: two rounds of workgroups with two columns a lane
    ones = how == "gates"
    q, k = (torch.randn(T, H * dk, generator=g).to(dtype) for _ in range(2))
    v = torch.randn(T, H, vc, generator=g).to(dtype)
    state = torch.randn(3, H, dk, vc + ones, generator=g)
    step, bias, rate = torch.randn(T, H, generator=g).to(dtype), torch.randn(H, generator=g) - 1.0, torch.randn(H, generator=g) * 0.5 - 1.0
    gates = torch.stack([torch.rand(T, H, generator=g) * 0.3 + 0.7, torch.rand(T, H, generator=g)], dim=2)
    head = torch.rand(H, generator=g) * 0.3 + 0.7
    d = lambda t: t.to(DEV)
    kw = {"gates": dict(gates=d(gates)), "silu": dict(head_decay=d(head), silu=True),
          "step": dict(step=d(step), step_bias=d(bias), decay_log=d(rate))}[how]

    def walk(a, b):
        cols = list(range(a, b)) + ([vc] if ones else [])
        st = d(state[..., cols].contiguous())
        o = kernels.linear_scan(d(q), d(k), d(v[..., a:b].reshape(T, -1).contiguous()), st, torch.arange(3, device=DEV), cu, H, dk, len(cols),
                                q_scale=dk ** -0.5, q_lens=lens, **({**kw, "value_cols": b - a} if ones else kw))
        return o.view(T, H, -1).cpu(), st.cpu()

    whole, st = walk(0, vc)
    for a in range(0, vc, 64):
        b = min(vc, a + 64)
        part, own = walk(a, b)
        assert torch.equal(whole[..., a:b], part[..., :b - a]) and torch.equal(st[..., a:b], own[..., :b - a])
        assert torch.equal(whole[..., vc:], part[..., b - a:]) and torch.equal(st[..., vc:], own[..., b - a:])

    x = step.double() + bias.double()
    size = torch.logaddexp(x, torch.zeros_like(x))
    decay = {"gates": gates[..., 0].double(), "silu": head.double().expand(T, H), "step": torch.exp(-torch.exp(rate.double()) * size)}[how]
    weight = {"gates": gates[..., 1].double(), "silu": torch.ones(T, H, dtype=torch.float64), "step": size}[how]
    act = torch.nn.functional.silu if how == "silu" else lambda t: t
    qd, kd = act(q.double()).view(T, H, dk), act(k.double()).view(T, H, dk)
    vd = torch.cat([act(v.double()), torch.ones(T, H, 1, dtype=torch.float64)], dim=2) if ones else act(v.double())
    for i, (a, b) in enumerate(((0, 1130), (1130, 1132), (1132, T))):
        ref, s = _plain(qd[a:b], kd[a:b], vd[a:b], decay[a:b], weight[a:b], state[i], dk ** -0.5)
        sizes, s_sizes = _plain(qd[a:b].abs(), kd[a:b].abs(), vd[a:b].abs(), decay[a:b], weight[a:b], state[i].abs(), dk ** -0.5)
        # float32 sums of dk products of a state that holds about 1 / (1 - decay) tokens' terms, each a few roundings old
        bound = (dk + 64) * 2.0 ** -23
        assert float(((whole[a:b].double() - ref).abs() / sizes).max()) < bound
        assert float(((st[i].double() - s).abs() / s_sizes).max()) < bound


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("H,dk,dv", [(8, 128, 256), (2, 100, 70)])
def test_a_portion_alone_and_beside_others(H, dk, dv, dtype):
    """What a request gets, and the state left in its slot, do not depend on the other portions of the step: the same bits."""
    from xinfer_amd import kernels
    g = torch.Generator().manual_seed(H + dk)
    lens = [300, 2, 129, 1030, 64, 2300]
    T, B = sum(lens), len(lens)
    q, k, v = (torch.randn(T, H * n, generator=g).to(dtype).to(DEV) for n in (dk, dk, dv))
    z, state = (torch.randn(T, H * dk, generator=g) + 1.5).to(DEV), torch.randn(B, H, dk, dv, generator=g).to(DEV)
    first = [sum(lens[:b]) for b in range(B)]

    def walk(rows):
        at = torch.cat([torch.arange(first[b], first[b] + lens[b]) for b in rows]).to(DEV)
        own = [lens[b] for b in rows]
        cu = torch.tensor([sum(own[:i]) for i in range(len(own) + 1)], dtype=torch.int32, device=DEV)
        st = state[rows].clone()
        o = kernels.linear_scan(q[at], k[at], v[at], st, torch.arange(len(rows), device=DEV), cu, H, dk, dv, z=z[at], tau=8.0,
                                q_scale=dk ** -0.5, q_lens=own)
        return dict(zip(rows, zip(o.split(own), st)))

    everyone = walk(list(range(B)))
    for rows in [[b] for b in range(B)] + [[2, 0], [3, 1, 0]]:
        for b, (o, s) in walk(rows).items():
            assert torch.equal(o, everyone[b][0]) and torch.equal(s, everyone[b][1]), (rows, lens[b])


@pytest.mark.parametrize("H,dk,dv,lens", [(2, 100, 70, [300, 5, 130]), (8, 64, 96, [1030, 127, 1]), (1, 128, 256, [129, 64])])
def test_last_chunks_of_a_few_tokens(H, dk, dv, lens):
    """Last chunks of one and two tokens and more, beside portions in one piece, against float64."""
    from xinfer_amd import kernels
    g = torch.Generator().manual_seed(H + dk)
    T, B = sum(lens), len(lens)
    q, k, v = (torch.randn(T, H * n, generator=g).to(torch.bfloat16) for n in (dk, dk, dv))
    z, state = torch.randn(T, H * dk, generator=g) + 1.5, torch.randn(B, H, dk, dv, generator=g)
    cu = [0] + torch.tensor(lens).cumsum(0).tolist()
    st = state.to(DEV)
    o = kernels.linear_scan(q.to(DEV), k.to(DEV), v.to(DEV), st, torch.arange(B, device=DEV), torch.tensor(cu, dtype=torch.int32, device=DEV),
                            H, dk, dv, z=z.to(DEV), tau=8.0, q_scale=dk ** -0.5, q_lens=lens).cpu().double().view(T, H, dv)
    a = torch.sigmoid(z.double()).pow(1 / 8.0).view(T, H, dk)
    qd, kd, vd = (t.double().view(T, H, -1) for t in (q, k, v))
    bound = (dk + 64) * 2.0 ** -23          # as above
    for b in range(B):
        S, size = state[b].double(), state[b].double().abs()
        for t in range(cu[b], cu[b + 1]):
            S = a[t][..., None] * S + kd[t][..., None] * vd[t][:, None]
            size = a[t][..., None] * size + (kd[t][..., None] * vd[t][:, None]).abs()
            ref, most = ((x * y[..., None]).sum(1) * dk ** -0.5 for x, y in ((S, qd[t]), (size, qd[t].abs())))
            assert float(((o[t] - ref).abs() / most).max()) < bound
        assert float(((st[b].cpu().double() - S).abs() / size).max()) < bound


@pytest.mark.parametrize("kind", ["z", "head", "step", "gates"])
@pytest.mark.parametrize("H,dk,dv,dtype", [(3, 256, 40, torch.bfloat16), (4, 100, 130, torch.float32), (5, 64, 64, torch.bfloat16), (2, 24, 70, torch.float32)])
def test_tokens_fetched_together(H, dk, dv, dtype, kind):
    """Portions that end anywhere in a group of tokens give the bits of their tokens one at a time, results and states."""
    from xinfer_amd import kernels
    g = torch.Generator().manual_seed(dk)
    lens = [1, 2, 3, 5, 8, 17, 31]
    T, B = sum(lens), len(lens)
    vc = dv - 1 if kind == "gates" else dv
    starts = [sum(lens[:b]) for b in range(B + 1)]
    q, k = (torch.randn(T, H * dk, generator=g).to(dtype).to(DEV) for _ in range(2))
    v = torch.randn(T, H * vc, generator=g).to(dtype).to(DEV)
    rows = {"z": dict(z=torch.randn(T, H * dk, generator=g).to(DEV)), "head": {}, "step": dict(step=torch.randn(T, H, generator=g).to(dtype).to(DEV)),
            "gates": dict(gates=torch.rand(T, H, 2, generator=g).to(DEV))}[kind]
    fixed = {"z": dict(z_bias=torch.randn(H * dk, generator=g).to(DEV), tau=4.0), "head": dict(head_decay=torch.rand(H, generator=g).to(DEV)),
             "step": dict(step_bias=torch.randn(H, generator=g).to(DEV), decay_log=torch.randn(H, generator=g).to(DEV)), "gates": {}}[kind]
    state = torch.randn(B, H, dk, dv, generator=g).to(DEV)
    st, one = state.clone(), state.clone()
    cu = torch.tensor(starts, dtype=torch.int32, device=DEV)
    out = kernels.linear_scan(q, k, v, st, torch.arange(B, device=DEV), cu, H, dk, dv, value_cols=vc, **rows, **fixed)
    for t in range(max(lens)):
        live = [b for b in range(B) if t < lens[b]]
        at = torch.tensor([starts[b] + t for b in live], device=DEV)
        o = kernels.linear_scan(q[at], k[at], v[at], one, torch.tensor(live, device=DEV), torch.arange(len(live) + 1, dtype=torch.int32, device=DEV), H, dk, dv,
                                value_cols=vc, **{n: r[at] for n, r in rows.items()}, **fixed)
        assert torch.equal(out[at], o), t
    assert torch.equal(st, one)
