"""GPU tests of the 16-byte copies behind head dims the kernels are not built
for: the same bits as the 2-byte copies, which the same rows take when they
start one element off a 16-byte boundary.  BSHD rows and head-major rows, head
dims around the built widths, and strides with room between the rows."""
import pytest

pytestmark = pytest.mark.gpu


def _rows(torch, cuda, g, B, S, H, D, head_major, shift):
    """The same values for any shift: [B, S, H, D] rows `shift` elements off 16 bytes."""
    x = torch.randn((B, S, H, D), generator=g, device=cuda, dtype=torch.bfloat16)
    shape = (B, H, S, D + 8) if head_major else (B, S, H, D + 8)
    room = torch.full(shape, float("nan"), device=cuda, dtype=torch.bfloat16)
    view = room.transpose(1, 2) if head_major else room
    view[..., shift:shift + D] = x
    return view[..., shift:shift + D]


@pytest.mark.parametrize("D,Dv", [(72, 72), (96, 80), (120, 128), (136, 136), (200, 248), (192, 64)])
@pytest.mark.parametrize("head_major", [False, True])
@pytest.mark.parametrize("B,S,Hq,Hkv", [(1, 1, 1, 1), (2, 77, 6, 2), (1, 300, 28, 4)])
def test_forward_row_copies(cuda, D, Dv, head_major, B, S, Hq, Hkv):
    import torch
    import cuda_llm_ops_amd as fg
    print(f"({D},{Dv}) head_major={head_major} B{B} S{S} Hq{Hq} Hkv{Hkv}", flush=True)
    got = []
    for shift in (0, 1):
        g = torch.Generator(device=cuda)
        g.manual_seed(D + S)
        q, k, v = (_rows(torch, cuda, g, B, S, h, d, head_major, shift) for h, d in ((Hq, D), (Hkv, D), (Hkv, Dv)))
        room = torch.full((B, S, Hq, Dv + 8), 7.0, device=cuda, dtype=torch.bfloat16)
        _, lse = fg.flash_gqa_forward_bshd(q, k, v, out=room[..., shift:shift + Dv])
        torch.cuda.synchronize()
        o = room[..., shift:shift + Dv].contiguous()
        assert torch.isfinite(o.float()).all()
        assert bool((room[..., :shift] == 7.0).all()) and bool((room[..., shift + Dv:] == 7.0).all())
        got.append((o, lse))
    assert torch.equal(got[0][0].view(torch.int16), got[1][0].view(torch.int16))
    assert torch.equal(got[0][1], got[1][1])
