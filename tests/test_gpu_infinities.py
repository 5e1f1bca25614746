"""An infinite V value in the newest FP32 token reaches its channel as that infinity, as in the reference's sum over
tokens: rows and partial slots that only fill up a ragged end must not add a zero times it (a NaN)."""
import numpy as np
import pytest
import torch

from gpu_helpers import attention_errors, attention_ok, dev, host, make_case

pytestmark = pytest.mark.gpu

# Hq, Hkv, D, FP32 tokens, blocks
MERGE = [
    (2, 2, 80, 16, 0),      # whole units, one slot: the merge has 12 slot groups of 20 channel quads
    (9, 3, 64, 32, 5),      # the infinity not in the last slot
    (2, 1, 240, 24, 3),     # three units, a slot; four groups of 60 quads
    (16, 2, 128, 32, 20),   # the matrix-core kernel's partials
]


def check(oracle, case, seed):
    from tritiercache_amd import _C

    Hq, Hkv, D, nd, nb = case
    args = list(make_case(oracle, Hq, Hkv, D, nd, nb, 16, False, "none", seed))
    V = args[2]
    V[-1, 0, 1], V[-1, Hkv - 1, D - 1] = np.inf, -np.inf
    Q, dK, dV, _, KP, KS, KZ, VP, VS, VZ, ids = (dev(x) if isinstance(x, np.ndarray) else x for x in args[:11])
    out, mw = torch.zeros((Hq, D), device="cuda"), torch.zeros(nd + nb * 16, device="cuda")
    _C.fused_attention_decode(Q, dK, dV, nd, KP, KS, KZ, VP, VS, VZ, ids, nb, Hq, Hkv, D, out, mw, 16, "fp32")
    torch.cuda.synchronize()
    ro, rmw = oracle.fused_attention_decode(*args)
    got, want = host(out), np.asarray(ro).reshape(Hq, D)
    inf = np.isinf(want)
    assert inf.sum() == 2 * (Hq // Hkv)  # one channel of the first and of the last KV head's queries
    assert np.array_equal(got[inf], want[inf]), (case, got[inf], want[inf])
    got, want = np.where(inf, 0, got), np.where(inf, 0, want)
    err = attention_errors(got, want, host(mw), rmw)
    assert attention_ok(err), (case, err)


@pytest.mark.parametrize("case", MERGE, ids=str)
def test_merge_adds_no_slot_twice(oracle, case):
    check(oracle, case, seed=2100 + MERGE.index(case))

# ragged ends of the VALU kernel's FP32 units
UNIT = [
    (9, 3, 64, 16 * 63 + 5, 0),   # 64 units, 16 slots (as many as the merge has groups)
    (2, 2, 80, 1, 0),
    (8, 8, 256, 8 * 31 + 1, 2),   # units of 8 tokens
    (4, 2, 128, 37, 3),           # short contexts of head_dim 128
    (5, 5, 16, 17, 0),
]


@pytest.mark.parametrize("case", UNIT, ids=str)
def test_fp32_unit_weighs_no_row_twice(oracle, case):
    check(oracle, case, seed=2200 + UNIT.index(case))
