"""The rows a prefill keeps in f32 (sinks, recent window, waiting room) and its counters, at the lengths where a tier
starts or ends, from prompts at and one float past a 16-byte boundary: bit for bit the oracle's state."""
import numpy as np
import pytest
import torch

from gpu_helpers import compare_state, gpu_engine_state
from oracle import synth

pytestmark = pytest.mark.gpu

S, R, MSL = 4, 24, 400


@pytest.mark.parametrize("hkv,d,kgs,fp16", [(2, 64, 16, True), (3, 16, 32, False), (5, 80, 16, False)])
@pytest.mark.parametrize("q_len", [0, 3, S, S + 1, S + R, S + R + 1, S + R + 32, S + R + 32 * 5 + 31, MSL])
def test_prefill_rows_and_state(oracle, hkv, d, kgs, fp16, q_len):
    from tritiercache_amd import _C

    k, v = synth.normal(71, 0, (q_len, hkv, d)), synth.normal(71, 1, (q_len, hkv, d))
    want = oracle.engine(2 * hkv, hkv, d, MSL, S, R, 0.1, 0.99, 8, kgs, fp16)
    want.prefill(k, v)
    for shift in (0, 1):
        eng = _C.TriTierCacheEngine(2 * hkv, hkv, d, MSL, S, R, 0.1, 0.99, 8, kgs, "fp16" if fp16 else "fp32")
        dk, dv = (torch.zeros(x.size + 1, device="cuda")[shift:shift + x.size] for x in (k, v))
        dk.copy_(torch.from_numpy(np.ascontiguousarray(k).reshape(-1)))
        dv.copy_(torch.from_numpy(np.ascontiguousarray(v).reshape(-1)))
        eng.prefill(dk, dv, q_len)
        compare_state(gpu_engine_state(eng), want.state(), (q_len, shift))


def test_prefills_past_the_packed_store_keep_its_blocks(oracle):
    """Prompts one after another until the packed store is reallocated: blocks, ids and counters stay the oracle's."""
    from tritiercache_amd import _C

    args = (4, 2, 32, 64, S, R, 0.1, 0.99, 8, 16)
    eng, want = _C.TriTierCacheEngine(*args, "fp32"), oracle.engine(*args, False)
    for i in range(4):
        n = S + R + 16 * 40 + 5
        k, v = synth.normal(73, 2 * i, (n, 2, 32)), synth.normal(73, 2 * i + 1, (n, 2, 32))
        eng.prefill(torch.from_numpy(k).cuda(), torch.from_numpy(v).cuda(), n)
        want.prefill(k, v)
        compare_state(gpu_engine_state(eng), want.state(), i)
