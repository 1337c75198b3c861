"""GPU tests of the ragged decode's even sharing of token blocks over teams of
workgroups, and of the combine's ways, where their bounds lie: empty sequences,
lengths around a 128-token block, fewer blocks than teams, one sequence over
most teams among short ones, more sequences than a workgroup has threads; and
uniform batches whose split count crosses the combine's 8, 32 and 128 partials.

Checked against float64 attention at the decode bar (max-abs 2e-2, mean-abs
2e-3) and, for the LSE (a sum of fp32 exponentials), 1e-3; in a workspace
filled with NaN bytes, so that a partial read before it is written shows.
"""
import math

import pytest

from tests._helpers import assert_close

pytestmark = pytest.mark.gpu

LENS = {
    "all_empty": [0, 0, 0],
    "one_token": [1],
    "block_edges": [128, 129, 127, 0, 1, 256, 0],
    "fewer_blocks_than_teams": [700, 0, 300],
    "one_long": [3, 20000, 0, 700, 129],
    "many_short": [(37 * i) % 301 for i in range(700)],
}


def _reference(q, k, v):
    """float64 attention of q [Hq, D] over k, v [S, Hkv, D] -> out, natural-log LSE."""
    import torch
    Hq, Hkv = q.shape[0], k.shape[1]
    qd = q.double().view(Hkv, Hq // Hkv, -1)
    s = torch.matmul(qd, k.double().permute(1, 2, 0).contiguous()) / math.sqrt(128)
    o = torch.matmul(torch.softmax(s, dim=2), v.double().permute(1, 0, 2).contiguous())
    return o.reshape(Hq, -1), torch.logsumexp(s, dim=2).reshape(Hq)


def _compare(out, lse, refs, what):
    import torch
    for b, (o_ref, l_ref) in enumerate(refs):
        if o_ref is None:
            assert torch.all(out[b] == 0) and torch.all(lse[b] == -math.inf), f"{what}: empty sequence {b}"
            continue
        assert_close(out[b].float().cpu().numpy(), o_ref.cpu().numpy(), f"{what}: sequence {b}")
        assert (lse[b].double() - l_ref).abs().max() <= 1e-3, f"{what}: lse of sequence {b}"


@pytest.mark.parametrize("heads", [(4, 1), (32, 2), (12, 3), (32, 8)])
@pytest.mark.parametrize("lens", list(LENS))
def test_ragged_teams(cuda, lens, heads):
    import torch
    import cuda_llm_ops_amd as fg
    n, (Hq, Hkv) = LENS[lens], heads
    B, S, page = len(n), max(max(n), 1), 16
    g = torch.Generator(device=cuda)
    g.manual_seed(B + Hq)
    per = -(-S // page)
    kc, vc = (torch.randn((B * per, page, Hkv, 128), generator=g, device=cuda, dtype=torch.bfloat16) for _ in range(2))
    q = torch.randn((B, Hq, 128), generator=g, device=cuda, dtype=torch.bfloat16)
    table = torch.randperm(B * per, generator=g, device=cuda).to(torch.int32).view(B, per)
    lens_d = torch.tensor(n, device=cuda, dtype=torch.int32)
    k8, v8 = kc.to(torch.float8_e4m3fn), vc.to(torch.float8_e4m3fn)

    def rows(cache, b):
        return cache[table[b].long()].reshape(per * page, Hkv, 128)[:n[b]]

    for kind in ("contiguous", "paged", "paged fp8"):
        what = f"{lens} heads={heads} {kind}"
        print(what, flush=True)
        lse = torch.full((B, Hq), 7.0, device=cuda)
        out = torch.full((B, Hq, 128), 7.0, device=cuda, dtype=torch.bfloat16)
        if kind == "contiguous":
            ws = torch.full((fg.decode_workspace_bytes(B, S, Hq, Hkv, ragged=True),), 255, device=cuda, dtype=torch.uint8)
            k = torch.full((B, S, Hkv, 128), math.nan, device=cuda, dtype=torch.bfloat16)
            v = k.clone()
            for b in range(B):
                k[b, :n[b]], v[b, :n[b]] = rows(kc, b), rows(vc, b)
            fg.decode_flash_gqa_bshd(q, k, v, out=out, seqlens=lens_d, lse=lse, workspace=ws)
        else:
            ws = torch.full((fg.paged_decode_workspace_bytes(B, S, Hq, Hkv, page),), 255, device=cuda, dtype=torch.uint8)
            ck, cv = (k8, v8) if "fp8" in kind else (kc, vc)
            fg.decode_flash_gqa_paged(q, ck, cv, table, lens_d, out=out, lse=lse, max_seqlen=S, workspace=ws)
        ck, cv = (k8, v8) if "fp8" in kind else (kc, vc)
        refs = [_reference(q[b], rows(ck, b), rows(cv, b)) if n[b] else (None, None) for b in range(B)]
        _compare(out, lse, refs, what)


@pytest.mark.parametrize("splits", [8, 9, 32, 33, 128, 129])
@pytest.mark.parametrize("heads", [(5, 5), (16, 1)])
def test_combine_ways(cuda, splits, heads):
    import torch
    import cuda_llm_ops_amd as fg
    (Hq, Hkv), S = heads, 128 * splits - 5
    print(f"splits={splits} heads={heads}", flush=True)
    g = torch.Generator(device=cuda)
    g.manual_seed(splits)
    k, v = (torch.randn((2, S, Hkv, 128), generator=g, device=cuda, dtype=torch.bfloat16) for _ in range(2))
    q = torch.randn((2, Hq, 128), generator=g, device=cuda, dtype=torch.bfloat16)
    ws = torch.full((fg.decode_workspace_bytes(2, S, Hq, Hkv, split_tokens=128),), 255, device=cuda, dtype=torch.uint8)
    lse = torch.empty((2, Hq), device=cuda)
    out = fg.decode_flash_gqa_bshd(q, k, v, lse=lse, split_tokens=128, workspace=ws)
    _compare(out, lse, [_reference(q[b], k[b], v[b]) for b in range(2)], f"splits={splits} heads={heads}")
