"""GPU tests of a scale of 0 (every visible score is 0): O is the mean of the
visible V rows and the LSE the log of their number, at lengths that end inside a
tile, where masked and visible keys meet in one step.

Bars: O 2e-2 maximum and 2e-3 mean against float64; the LSE 1e-5 (one fp32
logarithm of a sum of ones)."""
import math

import pytest

from tests._helpers import assert_close

pytestmark = pytest.mark.gpu


def _inputs(cuda, B, Sq, Skv, Hq, Hkv, dqk, dv):
    import torch
    g = torch.Generator(device=cuda)
    g.manual_seed(Sq + dqk)
    return (torch.randn(s, generator=g, device=cuda, dtype=torch.bfloat16)
            for s in ((B, Sq, Hq, dqk), (B, Skv, Hkv, dqk), (B, Skv, Hkv, dv)))


def _check_uniform(out, lse, v, visible, sink, what):
    """visible: bool [Sq, Skv]; sink: [Hq] or None."""
    import torch
    Hq, Hkv = out.shape[2], v.shape[2]
    n = visible.sum(1).double()                                                     # [Sq]
    s = torch.zeros(Hq, device=v.device, dtype=torch.float64) if sink is None else sink.double()
    total = n[None, :] + s[:, None]                                                 # [Hq, Sq]
    sums = torch.einsum("qk,bkhd->bqhd", visible.double().cpu(), v.double().cpu()).to(v.device)
    ref = sums.repeat_interleave(Hq // Hkv, dim=2) / total.t()[None, :, :, None]
    assert_close(out.float().cpu().numpy(), ref.cpu().numpy(), what)
    assert (lse.double() - torch.log(total)[None]).abs().max() <= 1e-5, f"{what}: lse"


@pytest.mark.parametrize("dqk,dv,kernel,window,with_sink", [
    (128, 128, "whole", 0, False), (128, 128, "split", 0, False), (128, 128, "wide", 0, False),
    (128, 128, "tall", 0, False), (128, 128, "whole", 70, True), (128, 128, "wide", 70, True),
    (192, 128, "whole", 0, False), (192, 128, "split", 0, False), (192, 128, "wide", 0, False),
    (64, 64, "whole", 0, False), (64, 64, "split", 0, False), (64, 64, "wide", 0, False), (64, 64, "whole", 70, True),
    (96, 80, "auto", 0, False), (256, 128, "auto", 0, False)])
@pytest.mark.parametrize("causal", [True, False])
def test_prefill_scale_zero(cuda, dqk, dv, kernel, window, with_sink, causal):
    import torch
    import cuda_llm_ops_amd as fg
    if window and not causal:
        causal, window = True, 0   # the sink without a window instead
    what = f"({dqk},{dv}) {kernel} causal={causal} window={window} sink={with_sink}"
    print(what, flush=True)
    S, Hq, Hkv = 300, 8, 2
    q, k, v = _inputs(cuda, 1, S, S, Hq, Hkv, dqk, dv)
    sink = torch.rand(Hq, device=cuda) + 0.5 if with_sink else None
    for scale in (0.0, -0.0):
        out, lse = fg.flash_gqa_forward_bshd(q, k, v, scale, causal=causal, window_size=window, sink=sink,
                                             kernel=kernel)
        i, j = torch.arange(S, device=cuda)[:, None], torch.arange(S, device=cuda)[None, :]
        visible = (j <= i) if causal else torch.ones((S, S), dtype=torch.bool, device=cuda)
        if window:
            visible = visible & (j > i - window)
        _check_uniform(out, lse, v, visible, sink, what)


def test_decode_scale_zero(cuda):
    import torch
    import cuda_llm_ops_amd as fg
    print("decode", flush=True)
    lens = [300, 77]
    q, k, v = _inputs(cuda, 2, 1, 300, 8, 2, 128, 128)
    for kw in ({}, {"split_tokens": 128}):
        lse = torch.empty((2, 8), device=cuda)
        out = fg.decode_flash_gqa_bshd(q[:, 0], k, v, 0.0, seqlens=torch.tensor(lens, device=cuda, dtype=torch.int32),
                                       lse=lse, **kw)
        for b, n in enumerate(lens):
            ref = v[b, :n].double().mean(0).repeat_interleave(4, dim=0)
            assert_close(out[b].float().cpu().numpy(), ref.cpu().numpy(), f"decode {kw} sequence {b}")
            assert (lse[b].double() - math.log(n)).abs().max() <= 1e-5
