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
