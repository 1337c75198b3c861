"""GPU test of a ragged decode's bits: with a given split length a sequence's
result does not depend on the rest of the batch; without one it may by
rounding, but every call on the same inputs gives the same bits."""
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("split_tokens", [0, 128, 1000])
@pytest.mark.parametrize("kind", ["contiguous", "paged", "paged fp8"])
def test_alone_and_among_others(cuda, kind, split_tokens):
    import torch
    import cuda_llm_ops_amd as fg
    print(f"{kind} split_tokens={split_tokens}", flush=True)
    lens, S, Hq, Hkv, page = [700, 0, 2500, 129, 1800, 1], 2500, 16, 2, 16
    B, per = len(lens), -(-2500 // page)
    g = torch.Generator(device=cuda)
    g.manual_seed(7)
    q = torch.randn((B, Hq, 128), generator=g, device=cuda, dtype=torch.bfloat16)
    kc, vc = (torch.randn((B * per, page, Hkv, 128), generator=g, device=cuda, dtype=torch.bfloat16) for _ in range(2))
    if "fp8" in kind:
        kc, vc = kc.to(torch.float8_e4m3fn), vc.to(torch.float8_e4m3fn)
    table = torch.arange(B * per, device=cuda, dtype=torch.int32).view(B, per)
    n = torch.tensor(lens, device=cuda, dtype=torch.int32)

    def call(rows):
        lse = torch.empty((len(rows), Hq), device=cuda)
        if kind == "contiguous":
            k, v = (x.view(B, -1, Hkv, 128)[rows, :S].contiguous() for x in (kc, vc))
            out = fg.decode_flash_gqa_bshd(q[rows].contiguous(), k, v, seqlens=n[rows].contiguous(), lse=lse,
                                           split_tokens=split_tokens)
        else:
            out = fg.decode_flash_gqa_paged(q[rows].contiguous(), kc, vc, table[rows].contiguous(),
                                            n[rows].contiguous(), lse=lse, max_seqlen=S, split_tokens=split_tokens)
        return out, lse

    every = list(range(B))
    out, lse = call(every)
    for _ in range(3):
        again = call(every)
        assert torch.equal(again[0], out) and torch.equal(again[1], lse)
    for b in every:
        o1, l1 = call([b])
        if split_tokens:
            assert torch.equal(o1[0], out[b]) and torch.equal(l1[0], lse[b]), f"sequence {b}"
        else:   # bf16 results of the same sums in another order
            assert (o1[0].float() - out[b].float()).abs().max() <= 2e-2
