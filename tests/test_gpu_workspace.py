"""The workspace size a caller asks for its longest context holds for every shorter one: contexts on both sides of the
line between the kernels, in one workspace, with and without mean weights. And the static scratch takes every call
that it can hold."""
import ctypes

import numpy as np
import pytest
import torch

from gpu_helpers import attention_errors, attention_ok, dev, host, make_case

pytestmark = pytest.mark.gpu

SHAPES = [(32, 32, 128), (16, 8, 128), (32, 8, 128), (24, 8, 128), (40, 10, 128), (40, 40, 128), (28, 4, 128),
          (8, 8, 128), (64, 64, 64), (32, 8, 64), (14, 2, 64), (9, 3, 64), (32, 32, 80), (16, 8, 256)]


@pytest.mark.parametrize("weights", [0, 1])
@pytest.mark.parametrize("kgs", [16, 32])
@pytest.mark.parametrize("shape", SHAPES, ids=str)
def test_size_grows_with_the_context(shape, kgs, weights):
    from tritiercache_amd import _lib

    q = _lib.load().tt_fused_attention_workspace_bytes
    for dense in ((0, 1, 5, 64, 260, 700, 2000), range(0, 2100, 60)):
        last = np.zeros(len(dense), np.int64)
        for blocks in [*range(0, 1200, 7), *range(1200, 9000, 61)]:
            need = np.array([q(d, blocks, *shape, kgs, weights) for d in dense])
            assert (np.diff(need) >= 0).all() and (need >= last).all() and need[0] > 0, (shape, blocks, need, last)
            last = need


@pytest.mark.parametrize("weights", [False, True])
@pytest.mark.parametrize("Hq,Hkv,D,nd,longest", [(32, 32, 128, 37, 300), (16, 8, 128, 21, 560), (64, 64, 64, 17, 480)])
def test_shorter_contexts_in_the_longest_ones_workspace(oracle, Hq, Hkv, D, nd, longest, weights):
    from tritiercache_amd import _lib

    L = _lib.load()
    args = make_case(oracle, Hq, Hkv, D, nd, longest, 16, False, "none", seed=2300 + Hq)
    Q, dK, dV, _, KP, KS, KZ, VP, VS, VZ, ids = (dev(x) if isinstance(x, np.ndarray) else x for x in args[:11])
    size = int(L.tt_fused_attention_workspace_bytes(nd, longest, Hq, Hkv, D, 16, int(weights)))
    ws = torch.empty(size, dtype=torch.uint8, device="cuda")
    stream = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    for blocks in (longest, longest - 1, *range(longest - 4, 0, -8), 0):
        out, mw = torch.zeros((Hq, D), device="cuda"), torch.zeros(nd + blocks * 16, device="cuda")
        rc = L.tt_fused_attention_decode_ws(Q.data_ptr(), dK.data_ptr(), dV.data_ptr(), nd, KP.data_ptr(), KS.data_ptr(),
                                            KZ.data_ptr(), VP.data_ptr(), VS.data_ptr(), VZ.data_ptr(), ids.data_ptr(),
                                            blocks, Hq, Hkv, D, out.data_ptr(), mw.data_ptr() if weights else None, 16, 0,
                                            ws.data_ptr(), size, stream)
        assert rc == 0, (blocks, L.tt_last_error())
        if blocks in (longest, longest - 20, 0):
            torch.cuda.synchronize()
            ro, rmw = oracle.fused_attention_decode(Q.cpu().numpy(), *args[1:11], blocks, *args[12:])
            err = attention_errors(host(out), ro, *((host(mw), rmw) if weights else ()))
            assert attention_ok(err), (blocks, err)


@pytest.mark.parametrize("D", [16, 80, 112, 144, 192, 208, 224, 256])
def test_noalloc_takes_what_fits_with_a_slot_per_head(D):
    """The largest context whose logits, row statistics and one partial slot per head fit the static scratch is taken
    by the _noalloc call, and one more block is not (no launch: the output's NULL pointer is refused after the
    scratch's check)."""
    from tritiercache_amd import _lib

    L = _lib.load()
    p, up = 0x10000, lambda x: (x + 255) & ~255  # noqa: E731
    for Hq, Hkv in ((8, 8), (24, 3), (12, 3), (20, 5), (40, 10), (80, 10), (56, 14), (160, 20), (160, 40)):
        def taken(nb):
            rc = L.tt_fused_attention_decode_noalloc(p, p, p, 0, p, p, p, p, p, p, p, nb, Hq, Hkv, D, None, p, 16, 0, None)
            assert rc == 1
            return "attn_output" in _lib.last_error()

        fixed = up(8 * Hq) + up(4 * Hq * D) + up(8 * Hq)
        nb = ((32 << 20) - fixed) // (4 * Hq * 16)
        assert taken(nb) and taken(nb - 30) and not taken(nb + 1), (Hq, Hkv, D, nb, _lib.last_error())
