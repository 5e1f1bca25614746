"""The VALU attention kernel (head dims other than 128, and 64 with an odd number of KV heads) and the merge, where a
wave holds several units: more work than one unit per wave of the launch, ragged tails of both kinds, and tiers and queries that
start one element past an aligned address."""
import numpy as np
import pytest
import torch

from gpu_helpers import attention_errors, attention_ok, dev, host, make_case

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def C():
    from tritiercache_amd import _C
    return _C


def _shifted(a):
    """The array on the GPU as a view one element past its allocation."""
    t = dev(a)
    base = torch.zeros(t.numel() + 1, dtype=t.dtype, device="cuda")
    base[1:].copy_(t.reshape(-1))
    return base[1:].view(t.shape)


CASES = [
    # Hq, Hkv, D, nd, nb, kgs, fp16, mask
    (64, 64, 80, 259, 130, 16, False, "tail"),    # several units per wave (64 heads share the device)
    (96, 48, 96, 33, 91, 32, True, "holes"),
    (16, 8, 256, 671, 300, 16, False, "block"),   # FP32 units of 8 tokens, a ragged last one
    (8, 1, 256, 9, 70, 32, True, "tail"),         # eight heads of 256 channels
    (9, 3, 64, 1, 700, 16, True, "holes"),        # more than 128 units per head
    (5, 5, 16, 1030, 0, 16, False, "none"),       # FP32 tokens only
    (10, 5, 240, 0, 37, 32, False, "tail"),       # packed tokens only
    (12, 3, 48, 17, 1, 16, True, "all"),
    (2, 1, 128, 40, 3300, 16, False, "holes"),    # one head over the device: more than 256 partial slots to merge
]


@pytest.mark.parametrize("shift", [False, True])
@pytest.mark.parametrize("case", CASES, ids=[str(c) for c in CASES])
def test_split_kernel_vs_oracle(C, oracle, case, shift):
    Hq, Hkv, D, nd, nb, kgs, fp16, mask = case
    args = make_case(oracle, Hq, Hkv, D, nd, nb, kgs, fp16, mask, seed=1700 + CASES.index(case))
    put = _shifted if shift else dev
    Q, dK, dV, _, KP, KS, KZ, VP, VS, VZ, ids = (put(x) if isinstance(x, np.ndarray) else x for x in args[:11])
    out = torch.full((Hq, D), float("nan"), device="cuda")
    mw = torch.full((nd + nb * kgs,), float("nan"), device="cuda")
    C.fused_attention_decode(Q, dK, dV, nd, KP, KS, KZ, VP, VS, VZ, ids, nb, Hq, Hkv, D, out, mw, kgs,
                             "fp16" if fp16 else "fp32")
    torch.cuda.synchronize()
    ro, rmw = oracle.fused_attention_decode(*args)
    err = attention_errors(host(out), ro, host(mw), rmw)
    assert attention_ok(err), (case, err)


def test_noalloc_plans_fewer_slots_where_the_scratch_is_short():
    """A call whose partials of the usual plan no longer fit beside its logits runs with half the slots; a call
    whose logits alone pass the scratch is still refused."""
    from tritiercache_amd import _lib

    L = _lib.load()
    Hq, Hkv, D, kgs = 8, 8, 256, 16
    need = lambda nb: L.tt_fused_attention_workspace_bytes(0, nb, Hq, Hkv, D, kgs, 1)  # noqa: E731
    limit = 32 << 20
    nb = max(n for n in range(60000, 65536, 16) if need(n) <= limit) + 256  # 128 KiB of logits past the fit
    assert need(nb) > limit
    g = torch.Generator(device="cuda").manual_seed(5)
    rnd = lambda *s: torch.randn(s, generator=g, device="cuda")  # noqa: E731
    words = lambda *s: torch.randint(-2**31, 2**31 - 1, s, generator=g, device="cuda", dtype=torch.int32)  # noqa: E731
    n = nb * kgs
    t = [rnd(Hq, D), None, None, words(nb, 1, Hkv, D), rnd(nb, Hkv, D).abs(), rnd(nb, Hkv, D), words(n, Hkv, D // 16),
         rnd(n, Hkv).abs(), rnd(n, Hkv), torch.arange(n, device="cuda")]
    p = [x.data_ptr() if x is not None else None for x in t]
    res = []
    for fn in (L.tt_fused_attention_decode, L.tt_fused_attention_decode_noalloc):
        out, mw = torch.zeros((Hq, D), device="cuda"), torch.zeros(n, device="cuda")
        rc = fn(*p[:3], 0, *p[3:], nb, Hq, Hkv, D, out.data_ptr(), mw.data_ptr(), kgs, 0, None)
        assert rc == 0, L.tt_last_error()
        torch.cuda.synchronize()
        res.append((host(out), host(mw)))
    err = attention_errors(res[1][0], res[0][0], res[1][1], res[0][1])
    assert attention_ok(err), err
    refused = L.tt_fused_attention_decode_noalloc(*p[:3], 0, *p[3:], 65600, Hq, Hkv, D, p[0], p[0], kgs, 0, None)
    assert refused == 1
