"""Launch sizes of the quantisers and dequantisers past the sizes that a test can allocate: no launch holds more
work-items than a dispatch counts (2^32), and none is left out (host arithmetic, compiled with g++)."""
import ctypes
import os
import shutil
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "tritiercache_amd", "csrc")
LIMIT = (1 << 32) - 1


@pytest.fixture(scope="module")
def grid(tmp_path_factory):
    if not shutil.which("g++"):
        pytest.skip("g++ not available")
    d = tmp_path_factory.mktemp("grid")
    (d / "g.cpp").write_text('#include "tt_quant_grid.h"\nextern "C" {\n'
                             "int k_slice(int nb, long long row) { return tt::quant_k_slice(nb, row); }\n"
                             "int k_fits(long long q) { return tt::deq_k_wide_fits(q); }\n"
                             "int v_fits(long long w) { return tt::deq_v_wide_fits(w); }\n"
                             "long long v_groups(long long w) { return tt::deq_v_wide_groups(w); }\n"
                             "int k_streams(long long v, int kgs, int f) { return tt::deq_k_streams(v, kgs, f); }\n"
                             "int v_streams(long long v, int d, int f) { return tt::deq_v_streams(v, d, f); }\n}\n")
    subprocess.run(["g++", "-shared", "-fPIC", "-std=c++17", "-I", CSRC, str(d / "g.cpp"), "-o", str(d / "g.so")],
                   check=True)
    L = ctypes.CDLL(str(d / "g.so"))
    L.v_groups.restype = ctypes.c_longlong
    return L


N = [1, 127, 128, 129, 65535, 65536, 1 << 30, (1 << 31) - 257, (1 << 31) - 129, (1 << 31) - 128, (1 << 31) - 127,
     (1 << 31) - 1, 1 << 31, (1 << 31) + 1, 3 << 30, LIMIT - 256, LIMIT]


@pytest.mark.parametrize("words", N)
def test_wide_v_launch_stays_within_a_dispatch(grid, words):
    w = ctypes.c_longlong(words)
    threads = 256 * grid.v_groups(w)
    assert threads >= 2 * words  # 4 quads of a word over 2 quads per thread
    assert bool(grid.v_fits(w)) == (threads <= LIMIT)


@pytest.mark.parametrize("quads", N)
def test_wide_k_launch_stays_within_a_dispatch(grid, quads):
    if grid.k_fits(ctypes.c_longlong(quads)):
        assert (quads + 255) // 256 * 256 <= LIMIT


@pytest.mark.parametrize("row", [16, 80, 1024, 4096, 32768, 1 << 20, (1 << 31) - 16])
def test_quantize_k_slices_cover_the_blocks(grid, row):
    for blocks in (1, 65535, 65536, LIMIT // row - 1, LIMIT // row, LIMIT // row + 1, (1 << 31) - 1):
        if not 0 < blocks < 1 << 31:
            continue
        per = grid.k_slice(blocks, ctypes.c_longlong(row))
        assert 1 <= per <= blocks and (per * row + 255) // 256 * 256 <= LIMIT
        # a slice is as large as a dispatch allows, so the launches are few and cover every block
        assert per == blocks or ((per + 1) * row + 255) // 256 * 256 > LIMIT - 256


@pytest.mark.parametrize("fp16", [0, 1])
@pytest.mark.parametrize("kgs,d", [(16, 64), (32, 80), (16, 256)])
def test_streaming_stores_start_past_the_last_level_cache(grid, kgs, d, fp16):
    for mib in range(64, 512):
        values, m = (mib << 20) // 4 // (kgs * d) * kgs * d, 2 if fp16 else 4
        total = lambda per: 4 * values + values // 4 + 2 * m * (values // per)  # noqa: E731
        v = ctypes.c_longlong(values)
        assert bool(grid.k_streams(v, kgs, fp16)) == (total(kgs) > (280 if fp16 else 256) << 20)
        assert bool(grid.v_streams(v, d, fp16)) == (total(d) > 256 << 20)
