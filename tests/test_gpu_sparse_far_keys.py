"""GPU tests of the sparse prefill where rows see many keys on average (more than
16384, half of them under the causal mask) and the grid is larger than two
workgroups per CU: two steps of rows in flight, lists of 257 to 512 entries
sorted by key.  Both sides of each line; lists whose usable entries make no
step, one, an odd and an even number; K and V rows of different strides.
Against the CPU oracle (2e-2 maximum and 2e-3 mean; LSE 1e-3)."""
import math

import numpy as np
import pytest

import oracle
from tests._helpers import assert_close, from_torch_bf16, to_torch_bf16

pytestmark = pytest.mark.gpu

SCALE = 1.0 / math.sqrt(128)


@pytest.mark.parametrize("Skv,causal", [(16384, False), (16385, False), (32769, True), (32770, True), (60000, False)])
@pytest.mark.parametrize("n", [255, 256, 257, 512, 513, 1100])
def test_sparse_far_keys(cuda, Skv, causal, n):
    import torch
    import cuda_llm_ops_amd as fg
    v_pad = 8 if (n + Skv) % 2 else 0
    print(f"Skv{Skv} causal={causal} n{n} v_pad={v_pad}", flush=True)
    Sq, H = 258, 8   # 2064 items of one head: 516 workgroups
    rng = np.random.default_rng(n + Skv)
    q = oracle.normal_bf16(n, (1, Sq, H, 128))
    k = oracle.normal_bf16(n, (1, Skv, H, 128), stream=1)
    v = oracle.normal_bf16(n, (1, Skv, H, 128), stream=2)
    qd, kd, vd = (to_torch_bf16(x, cuda) for x in (q, k, v))
    idx = rng.integers(0, Sq if causal else Skv, size=(1, H, Sq, n)).astype(np.int32)
    # usable entries of row i: none, 1, 32, 33, 64, 65, 96, 97, ..., all
    keep = np.array([0, 1, 32, 33, 64, 65, 96, 97, 224, n])[np.arange(Sq) % 10]
    order = rng.random(idx.shape).argsort(axis=-1)
    idx[order >= keep[None, None, :, None]] = -1
    if v_pad:
        wide = torch.zeros((1, Skv, H, 128 + v_pad), device=cuda, dtype=torch.bfloat16)
        wide[..., :128] = vd
        vd = wide[..., :128]
    out, lse = fg.flash_sgqa_forward_bshd(qd, kd, vd, torch.from_numpy(idx).to(cuda), SCALE, causal=causal)
    torch.cuda.synchronize()
    o_ref, l_ref = oracle.sparse_prefill(q, k, v, idx, SCALE, causal=causal)
    lse = lse.cpu().numpy()
    assert_close(oracle.bf16_to_f32(from_torch_bf16(out)), oracle.bf16_to_f32(o_ref), f"Skv{Skv} n{n}")
    fin = np.isfinite(l_ref)
    assert np.array_equal(np.isfinite(lse), fin)
    assert np.max(np.abs(lse[fin] - l_ref[fin]), initial=0.0) <= 1e-3
