"""GPU test of the sparse prefill at a scale of 0 (every visible score is 0): O
is the mean of the listed V rows and the LSE the log of their number, for lists
that end inside a 32-entry step, where masked and visible entries meet.

Bars: O 2e-2 maximum and 2e-3 mean against float64; the LSE 1e-5 (one fp32
logarithm of a sum of ones)."""
import math

import numpy as np
import pytest

from tests._helpers import assert_close

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [20, 33, 600])
@pytest.mark.parametrize("causal", [True, False])
def test_sparse_scale_zero(cuda, n, causal):
    import torch
    import cuda_llm_ops_amd as fg
    print(f"sparse n={n} causal={causal}", flush=True)
    Sq, Skv, Hq, Hkv = 50, 900, 8, 2
    g = torch.Generator(device=cuda)
    g.manual_seed(n)
    q, k, v = (torch.randn((1, s, h, 128), generator=g, device=cuda, dtype=torch.bfloat16)
               for s, h in ((Sq, Hq), (Skv, Hkv), (Skv, Hkv)))
    rng = np.random.default_rng(n)
    idx = np.stack([[rng.permutation(Skv)[:n] for _ in range(Sq)] for _ in range(Hkv)])[None].astype(np.int32)
    if causal:
        idx[0, :, :, 0] = 0   # every row sees a key
    out, lse = fg.flash_sgqa_forward_bshd(q, k, v, torch.from_numpy(idx).to(cuda), 0.0, causal=causal)
    out, lse, vd = out.double().cpu().numpy(), lse.double().cpu().numpy(), v.double().cpu().numpy()
    for r in range(Sq):
        for h in range(Hq):
            keys = [j for j in idx[0, h // (Hq // Hkv), r] if not causal or j <= r]
            assert_close(out[0, r, h], vd[0, keys, h // (Hq // Hkv)].mean(0), f"row {r} head {h}")
            assert abs(lse[0, h, r] - math.log(len(keys))) <= 1e-5, f"lse of row {r} head {h}"
