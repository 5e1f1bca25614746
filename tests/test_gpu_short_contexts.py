"""Head dims 128 and 64 on both sides of the line between the VALU kernel (short contexts) and the matrix cores, with
ragged and masked tails in both block lengths: output and mean weights against the oracle."""
import numpy as np
import pytest
import torch

from gpu_helpers import attention_errors, attention_ok, dev, host, make_case

pytestmark = pytest.mark.gpu

# Hq, Hkv, D, FP32 tokens, k_group_size, fp16, mask, blocks below and above the line
SHAPES = [
    (32, 32, 128, 37, 16, False, "holes", 265, 285),
    (32, 16, 128, 21, 32, True, "tail", 119, 131),
    (32, 8, 128, 50, 16, False, "block", 133, 147),
    (24, 8, 128, 33, 32, True, "tail", 67, 75),
    (28, 4, 128, 9, 16, False, "holes", 1, 40),
    (64, 64, 64, 17, 16, True, "tail", 105, 117),
    (32, 8, 64, 21, 16, False, "holes", 505, 520),
    (24, 8, 64, 9, 32, True, "block", 250, 263),
    (14, 2, 64, 20, 16, False, "tail", 180, 200),
]


@pytest.mark.parametrize("above", [False, True])
@pytest.mark.parametrize("shape", SHAPES, ids=[str(s[:7]) for s in SHAPES])
def test_both_kernels_vs_oracle(oracle, shape, above):
    from tritiercache_amd import _C

    hq, hkv, d, nd, kgs, fp16, mask = shape[:7]
    nb = shape[7 + above]
    args = make_case(oracle, hq, hkv, d, nd, nb, kgs, fp16, mask, seed=1900 + nb, k_outliers=True)
    Q, dK, dV, _, KP, KS, KZ, VP, VS, VZ, ids = (dev(x) if isinstance(x, np.ndarray) else x for x in args[:11])
    out = torch.full((hq, d), float("nan"), device="cuda")
    mw = torch.full((nd + nb * kgs,), float("nan"), device="cuda")
    _C.fused_attention_decode(Q, dK, dV, nd, KP, KS, KZ, VP, VS, VZ, ids, nb, hq, hkv, d, out, mw, kgs,
                              "fp16" if fp16 else "fp32")
    torch.cuda.synchronize()
    ro, rmw = oracle.fused_attention_decode(*args)
    err = attention_errors(host(out), ro, host(mw), rmw)
    assert attention_ok(err), (shape, nb, err)
