"""GPU tests of a sliding window longer than the sequence, up to the largest
value the argument holds: the same bits as a window of the sequence's length
(every causal key is visible either way), forward and backward."""
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("window", [5000, (1 << 30) + 3, (1 << 31) - 1])
@pytest.mark.parametrize("B,Sq,Skv,Hq,Hkv", [(1, 300, 300, 8, 1), (2, 130, 257, 4, 4), (1, 700, 200, 4, 2)])
def test_window_past_the_sequence(cuda, window, B, Sq, Skv, Hq, Hkv):
    import torch
    import cuda_llm_ops_amd as fg
    print(f"window={window} B{B} Sq{Sq} Skv{Skv} Hq{Hq} Hkv{Hkv}", flush=True)
    g = torch.Generator(device=cuda)
    g.manual_seed(Sq)
    q, k, v, do = (torch.randn(s, generator=g, device=cuda, dtype=torch.bfloat16)
                   for s in ((B, Sq, Hq, 128), (B, Skv, Hkv, 128), (B, Skv, Hkv, 128), (B, Sq, Hq, 128)))
    sink = torch.rand(Hq, generator=g, device=cuda) + 0.5

    def run(w):
        o, lse = fg.flash_gqa_forward_bshd(q, k, v, window_size=w, sink=sink, kernel="whole")
        return (o, lse, *fg.flash_gqa_backward_bshd(q, k, v, o, lse, do, window_size=w, dq_kernel="whole"),
                *fg.flash_gqa_backward_bshd(q, k, v, o, lse, do, window_size=w, dq_kernel="split"))

    want, got = run(max(Sq, Skv)), run(window)
    assert float(want[4].float().abs().max()) > 0
    for name, a, b in zip(("o", "lse", "dq", "dk", "dv", "dq split", "dk split", "dv split"), got, want):
        assert torch.equal(a, b), name
