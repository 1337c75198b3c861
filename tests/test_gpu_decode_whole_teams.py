"""GPU tests of ragged decodes whose sequences are of nearly one length, where a
team of workgroups takes whole sequences and leaves nothing to combine, on both
sides of that rule (with 8 KV heads there are 64 teams; a team may run up to 4
blocks of 128 tokens above an even share; not with a block per team or less):
one and two sequences per team, a last team with fewer, empty sequences among
the others, and the first lengths that are cut instead.

Against float64 at the decode bars (2e-2 maximum, 2e-3 mean; LSE 1e-3), in a
workspace filled with NaN bytes."""
import math

import pytest

from tests._helpers import assert_close

pytestmark = pytest.mark.gpu

LENS = {
    "a block per team": [256] * 32,
    "one sequence per team": [256] * 33,
    "one each, full": [700] * 64,
    "two per team": [256] * 65,
    "last team short": [300] * 127,
    "empty among them": [0 if i % 5 == 2 else 500 - i for i in range(64)],
    "only just even": [8 * 128] * 32,           # 8 blocks against an even share of 4
    "not even any more": [9 * 128] + [8 * 128] * 31,
    "three per team": [130 + i for i in range(129)],
}


@pytest.mark.parametrize("kind", ["contiguous", "paged", "paged fp8"])
@pytest.mark.parametrize("heads", [(32, 8), (8, 8)])
@pytest.mark.parametrize("lens", list(LENS))
def test_whole_sequences_per_team(cuda, lens, heads, kind):
    import torch
    import cuda_llm_ops_amd as fg
    print(f"{lens} heads={heads} {kind}", flush=True)
    n, (Hq, Hkv), page = LENS[lens], heads, 16
    B, S = len(n), max(n)
    g = torch.Generator(device=cuda)
    g.manual_seed(B + S)
    per = -(-S // page)
    kc, vc = (torch.randn((B * per, page, Hkv, 128), generator=g, device=cuda, dtype=torch.bfloat16) for _ in range(2))
    q = torch.randn((B, Hq, 128), generator=g, device=cuda, dtype=torch.bfloat16)
    lens_d = torch.tensor(n, device=cuda, dtype=torch.int32)
    lse = torch.full((B, Hq), 7.0, device=cuda)
    out = torch.full((B, Hq, 128), 7.0, device=cuda, dtype=torch.bfloat16)
    if kind == "contiguous":
        k, v = kc.view(B, -1, Hkv, 128)[:, :S], vc.view(B, -1, Hkv, 128)[:, :S]
        ws = torch.full((fg.decode_workspace_bytes(B, S, Hq, Hkv, ragged=True),), 255, device=cuda, dtype=torch.uint8)
        fg.decode_flash_gqa_bshd(q, k, v, out=out, seqlens=lens_d, lse=lse, workspace=ws)
    else:
        if "fp8" in kind:
            kc, vc = kc.to(torch.float8_e4m3fn), vc.to(torch.float8_e4m3fn)
        table = torch.randperm(B * per, generator=g, device=cuda).to(torch.int32).view(B, per)
        ws = torch.full((fg.paged_decode_workspace_bytes(B, S, Hq, Hkv, page),), 255, device=cuda, dtype=torch.uint8)
        fg.decode_flash_gqa_paged(q, kc, vc, table, lens_d, out=out, lse=lse, max_seqlen=S, workspace=ws)
        k, v = (c.view(torch.uint8 if "fp8" in kind else c.dtype)[table.long()].view(c.dtype).reshape(B, -1, Hkv, 128)
                for c in (kc, vc))
    for b, m in enumerate(n):
        if m == 0:
            assert torch.all(out[b] == 0) and torch.all(lse[b] == -math.inf), f"empty sequence {b}"
            continue
        s = torch.matmul(q[b].double().view(Hkv, Hq // Hkv, 128),
                         k[b, :m].double().permute(1, 2, 0).contiguous()) / math.sqrt(128)
        ref = torch.matmul(torch.softmax(s, dim=2), v[b, :m].double().permute(1, 0, 2).contiguous()).reshape(Hq, 128)
        assert_close(out[b].float().cpu().numpy(), ref.cpu().numpy(), f"sequence {b}")
        assert (lse[b].double() - torch.logsumexp(s, dim=2).reshape(Hq)).abs().max() <= 1e-3, f"lse of sequence {b}"
