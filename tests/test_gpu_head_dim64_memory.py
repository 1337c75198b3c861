"""GPU test of the device memory that prefills at head dims up to 64 hold: none
where they run on the tensors themselves and merge nothing; a workspace of the
stream's own, never the library's shared buffer, where the copies are made."""
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("causal", [True, False])
@pytest.mark.parametrize("D", [64, 40])
def test_no_scratch_in_place(cuda, D, causal):
    import torch
    import cuda_llm_ops_amd as fg
    from cuda_llm_ops_amd import flash_gqa as impl
    print(f"D={D} causal={causal}", flush=True)
    B, S, Hq, Hkv = 2, 4096, 16, 16
    copies = B * S * (2 * Hq + 2 * Hkv) * 128 * 2
    g = torch.Generator(device=cuda)
    g.manual_seed(D)
    q, k, v = (torch.randn((B, S, h, D), generator=g, device=cuda, dtype=torch.bfloat16) for h in (Hq, Hkv, Hkv))
    out, lse = torch.empty_like(q), torch.empty((B, Hq, S), device=cuda)
    impl._PREFILL_WORKSPACES.clear()

    def held(call):
        """Bytes that torch, and the device, hold more after the call."""
        torch.cuda.synchronize()
        t0, d0 = torch.cuda.memory_allocated(), torch.cuda.mem_get_info()[0] + torch.cuda.memory_reserved()
        keep = call()
        torch.cuda.synchronize()
        t1, d1 = torch.cuda.memory_allocated(), torch.cuda.mem_get_info()[0] + torch.cuda.memory_reserved()
        return t1 - t0, d0 - d1, keep

    held(lambda: fg.flash_gqa_forward_bshd(q, k, v, out=out, lse=lse, causal=causal))   # code objects are loaded
    mine, device, _ = held(lambda: fg.flash_gqa_forward_bshd(q, k, v, out=out, lse=lse, causal=causal))
    assert mine == 0 and device < 1 << 22
    mine, device, _p = held(lambda: fg.prepare_prefill(q, k, v, out=out, lse=lse, causal=causal))
    assert mine < 1 << 20 and device < 1 << 22
    # O over V, and unaligned rows: copies, in a workspace of torch's
    want = out.clone()
    vv = v.clone()
    mine, device, _ = held(lambda: fg.flash_gqa_forward_bshd(q, k, vv, out=vv, lse=lse, causal=causal))
    assert mine >= copies and device < 1 << 22
    assert (vv.float() - want.float()).abs().max() <= 2e-2
    impl._PREFILL_WORKSPACES.clear()
    room = torch.empty((B, S, Hq, D + 3), device=cuda, dtype=torch.bfloat16)
    mine, device, _ = held(lambda: fg.flash_gqa_forward_bshd(q, k, v, out=room[..., :D], lse=lse, causal=causal))
    assert mine >= copies and device < 1 << 22
    impl._PREFILL_WORKSPACES.clear()


@pytest.mark.parametrize("causal", [True, False])
def test_no_query_rows(cuda, causal):
    """Nothing to do, with keys enough that the size query is over 32 MB."""
    import torch
    import cuda_llm_ops_amd as fg
    print(f"causal={causal}", flush=True)
    q = torch.empty((1, 0, 16, 64), device=cuda, dtype=torch.bfloat16)
    k = torch.zeros((1, 8192, 16, 64), device=cuda, dtype=torch.bfloat16)
    out, lse = fg.flash_gqa_forward_bshd(q, k, k, causal=causal)
    torch.cuda.synchronize()
    assert out.shape == (1, 0, 16, 64) and lse.shape == (1, 16, 0)
