"""The heavy-hitter threshold (an exact k-th smallest score) at the candidate counts where its kernels change, over
scores that share digits, repeat, or differ in sign: an evicted token whose score equals the threshold becomes a heavy
hitter, one whose score is the next float below does not."""
import numpy as np
import pytest
import torch

from gpu_helpers import compare_state, gpu_engine_state
from oracle import synth

pytestmark = pytest.mark.gpu

S, R, RATIO = 4, 16, np.float32(0.1)


def _scores(kind, n):
    if kind == "zeros":
        return np.zeros(n, np.float32)
    if kind == "few":
        return np.resize(np.array([0.0, 1e-4, 1e-4, 3e-5, 0.5], np.float32), n)
    x = synth.normal(81, n % 97, (n,)).astype(np.float32)
    return x * np.float32(1e-3) if kind == "signed" else np.abs(x) ** 4 * np.float32(1e-5)


@pytest.mark.parametrize("kind", ["zeros", "few", "signed", "decayed"])
@pytest.mark.parametrize("n", [1, 64, 1025, 16385, 28672, 28673, 32768, 32769, 40001])
def test_threshold_is_exact(oracle, n, kind):
    from tritiercache_amd import _C

    q_len = S + R + n
    args = (2, 1, 16, q_len + 64, S, R, float(RATIO), 1.0, 8, 16)
    k, v = synth.normal(82, 0, (q_len, 1, 16)), synth.normal(82, 1, (q_len, 1, 16))
    dk, dv = torch.from_numpy(k).cuda(), torch.from_numpy(v).cuda()
    for below in (False, True):
        eng, want = _C.TriTierCacheEngine(*args, "fp32"), oracle.engine(*args, False)
        eng.prefill(dk, dv, q_len)
        want.prefill(k, v)
        vis = eng.visible()
        w = _scores(kind, vis)
        # scores of the candidates: the packed tokens' weights, zero in the waiting room
        cand = np.zeros(n, np.float32)
        cand[: n // 16 * 16] = w[S + R:]
        pick = int(np.float32(1.0 - RATIO) * np.float32(n - 1))
        thr = np.partition(cand, pick)[pick]
        w[S] = np.nextafter(thr, np.float32(-np.inf), dtype=np.float32) if below else thr  # the token evicted next
        eng.feedback(torch.from_numpy(w).cuda())
        want.feedback(w)
        eng.ingest(dk[0], dv[0])
        want.ingest(k[0], v[0])
        st = gpu_engine_state(eng)
        assert st["counters"]["hh_count"] == (0 if below else 1), (n, kind, below)
        compare_state(st, want.state(), (n, kind, below))
