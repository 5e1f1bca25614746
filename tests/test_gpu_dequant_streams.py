"""The dequantisers on both sides of the size from which their stores bypass the caches, with a ragged last workgroup:
bit for bit what the narrow kernels write (an output one float past a 16-byte boundary), which are held to the oracle
at small sizes; the first and last block, token and 65,536th block against the oracle too (the narrow K launch is
sliced after 65,535 blocks)."""
import numpy as np
import pytest
import torch

from gpu_helpers import host, same_bits

pytestmark = pytest.mark.gpu


def _words(g, *shape):
    return torch.randint(-2**31, 2**31 - 1, shape, generator=g, device="cuda", dtype=torch.int32)


def _meta(g, shape, fp16):
    x = torch.randn(shape, generator=g, device="cuda")
    return x.to(torch.float16).view(torch.uint16) if fp16 else x


def _same(a, b):
    return torch.equal(a.view(torch.int32), b.view(torch.int32))


# output MiB: below and above the line (256 MiB of tiers and output, 280 for K with FP16 metadata)
@pytest.mark.parametrize("mib", [180, 290])
@pytest.mark.parametrize("fp16", [False, True])
@pytest.mark.parametrize("h,d,kgs", [(1, 64, 16), (3, 80, 32)])
def test_wide_stores_match_narrow_ones(oracle, h, d, kgs, fp16, mib):
    from tritiercache_amd import _C

    g = torch.Generator(device="cuda").manual_seed(mib + d)
    nb = (mib << 20) // (4 * h * d * kgs) | 1  # an odd count: the last workgroup is ragged
    n, meta = nb * kgs, "fp16" if fp16 else "fp32"
    wide, narrow = torch.zeros(n * h * d, device="cuda"), torch.zeros(n * h * d + 1, device="cuda")[1:]
    kp, ks, kz = _words(g, nb, kgs // 16, h, d), _meta(g, (nb, h, d), fp16), _meta(g, (nb, h, d), fp16)
    for out in (wide, narrow):
        _C.dequantize_k(kp, ks, kz, out, nb, h, d, kgs, meta)
    assert _same(wide, narrow)
    for b in {0, nb - 1, min(65535, nb - 1)}:
        p, s, z = (host(t[b:b + 1]) for t in (kp, ks, kz))
        want = np.asarray(oracle.dequantize_k(p, s, z, 1, h, d, kgs, fp16)).reshape(-1)
        assert same_bits(host(wide[b * kgs * h * d:(b + 1) * kgs * h * d]), want), b
    wide.zero_(), narrow.zero_()
    vp, vs, vz = _words(g, n, h, d // 16), _meta(g, (n, h), fp16), _meta(g, (n, h), fp16)
    for out in (wide, narrow):
        _C.dequantize_v(vp, vs, vz, out, n, h, d, meta)
    assert _same(wide, narrow)
    for t in (0, n - 1):
        p, s, z = (host(x[t:t + 1]) for x in (vp, vs, vz))
        want = np.asarray(oracle.dequantize_v(p, s, z, 1, h, d, fp16)).reshape(-1)
        assert same_bits(host(wide[t * h * d:(t + 1) * h * d]), want), t
