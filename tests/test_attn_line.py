"""Which contexts the VALU attention kernel takes from the matrix cores (host arithmetic, compiled with g++), and that the
GPU tests of the two kernels' seam sit on both sides of it."""
import os
import shutil
import subprocess
import ctypes

import pytest

from test_gpu_short_contexts import SHAPES

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "tritiercache_amd", "csrc")
CUS = 256  # of an MI355X


@pytest.fixture(scope="module")
def line(tmp_path_factory):
    if not shutil.which("g++"):
        pytest.skip("g++ not available")
    d = tmp_path_factory.mktemp("line")
    (d / "l.cpp").write_text('#include "tt_attn_line.h"\nextern "C" {\n'
                             "int valu(int nd, int nb, int hq, int hkv, int d, int kgs, int cus) "
                             "{ return tt::use_valu(nd, nb, hq, hkv, d, kgs, cus); }\n"
                             "long long units(int hq, int hkv, int d, int cus) "
                             "{ return tt::short_units(hq, hkv, d, cus); }\n}\n")
    subprocess.run(["g++", "-shared", "-fPIC", "-std=c++17", "-I", CSRC, str(d / "l.cpp"), "-o", str(d / "l.so")],
                   check=True)
    L = ctypes.CDLL(str(d / "l.so"))
    L.units.restype = ctypes.c_longlong
    return L


@pytest.mark.parametrize("shape", SHAPES, ids=[str(s[:7]) for s in SHAPES])
def test_the_seam_tests_sit_on_both_sides(line, shape):
    hq, hkv, d, nd, kgs = shape[:5]
    below, above = (bool(line.valu(nd, nb, hq, hkv, d, kgs, CUS)) for nb in shape[7:])
    # more than four query heads per KV head of 128 channels: the matrix cores at any length
    assert (below, above) == ((False, False) if d == 128 and hq > 4 * hkv else (True, False)), shape


@pytest.mark.parametrize("hq,hkv,d", [(32, 32, 128), (16, 8, 128), (32, 8, 128), (64, 64, 64), (32, 8, 64), (14, 2, 64)])
@pytest.mark.parametrize("kgs", [16, 32])
def test_the_line_is_the_last_unit(line, hq, hkv, d, kgs):
    units, w = int(line.units(hq, hkv, d, CUS)), kgs // 16
    assert units > 0
    for dense in (0, 1, 16, 17):
        t = (dense + 15) // 16
        nb = (units - t) // w
        assert line.valu(dense, nb, hq, hkv, d, kgs, CUS) and not line.valu(dense, nb + 1, hq, hkv, d, kgs, CUS)


@pytest.mark.parametrize("hq,hkv,d", [(9, 3, 64), (32, 32, 80), (16, 8, 256), (8, 8, 16)])
def test_other_head_dims_are_the_valu_kernels(line, hq, hkv, d):
    assert line.valu(100000, 1000000, hq, hkv, d, 16, CUS)
