"""tt_engine_buffer waits for the stream: when it returns, what was enqueued there has run, so the pointer can be read
from any stream."""
import ctypes

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("which", range(20))
def test_buffer_waits_for_the_stream(which):
    from tritiercache_amd import _C, _lib

    L = _lib.load()
    eng = _C.TriTierCacheEngine(4, 2, 64, 256, 4, 16, 0.1, 0.99, 8, 16, "fp32")
    x = torch.randn((4096, 4096), device="cuda")
    torch.cuda.synchronize()
    side = torch.cuda.Stream()
    p, n, es = ctypes.c_void_p(), ctypes.c_int64(), ctypes.c_int()
    with torch.cuda.stream(side):
        for _ in range(20):  # some milliseconds
            y = x @ x
        done = torch.cuda.Event()
        done.record(side)
        assert not done.query()  # still running: else the test shows nothing
        _lib.check(L.tt_engine_buffer(eng._h, which, ctypes.byref(p), ctypes.byref(n), ctypes.byref(es),
                                      ctypes.c_void_p(side.cuda_stream)))
        assert done.query(), which
    del y
