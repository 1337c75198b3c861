"""GPU tests of the kernels built for head dim 64 (both head dims up to 64 and
multiples of 8, aligned): the same bits as the general path on zero-padded
copies, which the same inputs take when the output's rows are not 16-byte
aligned.  Lengths end inside a tile and a query block; every kernel shape the
two paths share; the unit pairs that merge through device memory, the
persistent grid and more units than CUs."""
import pytest

pytestmark = pytest.mark.gpu


def _both(cuda, B, Sq, Skv, Hq, Hkv, dqk, dv, **kw):
    import torch
    import cuda_llm_ops_amd as fg
    g = torch.Generator(device=cuda)
    g.manual_seed(Sq + dqk + dv)
    q, k, v = (torch.randn(s, generator=g, device=cuda, dtype=torch.bfloat16)
               for s in ((B, Sq, Hq, dqk), (B, Skv, Hkv, dqk), (B, Skv, Hkv, dv)))
    out, lse = fg.flash_gqa_forward_bshd(q, k, v, **kw)
    wide = torch.full((B, Sq, Hq, dv + 3), 7.0, device=cuda, dtype=torch.bfloat16)
    # (AUTO may choose another kernel shape for the copies)
    kw2 = dict(kw, kernel=fg.prefill_kernel_choice(q, k, v, **kw))
    out2, lse2 = fg.flash_gqa_forward_bshd(q, k, v, out=wide[..., :dv], **kw2)
    torch.cuda.synchronize()
    assert torch.isfinite(out.float()).all()
    assert torch.equal(out.view(torch.int16), out2.contiguous().view(torch.int16))
    assert torch.equal(lse, lse2)
    # and O into a strided view: nothing past its columns is written
    room = torch.full((B, Sq, Hq, dv + 8), 7.0, device=cuda, dtype=torch.bfloat16)
    fg.flash_gqa_forward_bshd(q, k, v, out=room[..., :dv], **kw)
    assert torch.equal(room[..., :dv].contiguous().view(torch.int16), out.view(torch.int16))
    assert bool((room[..., dv:] == 7.0).all())


@pytest.mark.parametrize("kernel", ["auto", "whole", "split", "wide"])
@pytest.mark.parametrize("dqk,dv", [(64, 64), (8, 8), (24, 64), (64, 40)])
@pytest.mark.parametrize("B,Sq,Skv,Hq,Hkv,causal", [(1, 333, 333, 8, 1, True), (2, 100, 257, 3, 3, False),
                                                     (1, 1, 1, 2, 1, True), (1, 130, 64, 4, 1, True)])
def test_native64_bits(cuda, kernel, dqk, dv, B, Sq, Skv, Hq, Hkv, causal):
    print(f"({dqk},{dv}) kernel={kernel} Sq{Sq} Skv{Skv} Hq{Hq} Hkv{Hkv} causal={causal}", flush=True)
    _both(cuda, B, Sq, Skv, Hq, Hkv, dqk, dv, causal=causal, kernel=kernel)


@pytest.mark.parametrize("S,Hq,Hkv", [(4096, 16, 1), (2049, 32, 8), (1030, 40, 8)])
def test_native64_large_grids(cuda, S, Hq, Hkv):
    print(f"S={S} Hq={Hq} Hkv={Hkv}", flush=True)
    _both(cuda, 1, S, S, Hq, Hkv, 64, 64)


@pytest.mark.parametrize("kernel,window", [("whole", 96), ("wide", 96), ("auto", 1600), ("wide", 0)])
def test_native64_window_and_sink(cuda, kernel, window):
    import torch
    print(f"kernel={kernel} window={window}", flush=True)
    sink = torch.rand(8, device=cuda) + 0.1
    for S in (700, 3000):
        _both(cuda, 1, S, S, 8, 2, 64, 48, window_size=window, sink=sink, kernel=kernel)
