"""GPU tests of prefills at head dims up to 64 that write O over one of their own
inputs: the same bits as into a tensor of its own, as for the other head dims
that run on copies."""
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("over", ["q", "k", "v", "v shifted"])
@pytest.mark.parametrize("D", [64, 40, 96])
@pytest.mark.parametrize("causal", [True, False])
def test_output_over_an_input(cuda, over, D, causal):
    import torch
    import cuda_llm_ops_amd as fg
    print(f"over={over} D={D} causal={causal}", flush=True)
    B, S, H = 2, 1700, 8
    g = torch.Generator(device=cuda)
    g.manual_seed(D)
    rows = B * S * H * D
    buf = {x: torch.randn(rows + 512 * D, generator=g, device=cuda, dtype=torch.bfloat16) for x in "qkv"}
    t = {x: buf[x][:rows].view(B, S, H, D) for x in "qkv"}
    # (the kernel that the copies take, so that the bits can be compared)
    room = torch.empty((B, S, H, D + 3), device=cuda, dtype=torch.bfloat16)
    want, want_lse = fg.flash_gqa_forward_bshd(t["q"], t["k"], t["v"], out=room[..., :D], causal=causal)
    want = want.contiguous()
    at = 512 * D if "shifted" in over else 0
    out = buf[over[0]][at:at + rows].view(B, S, H, D)
    _, lse = fg.flash_gqa_forward_bshd(t["q"], t["k"], t["v"], out=out, causal=causal)
    assert torch.equal(out, want) and torch.equal(lse, want_lse)
