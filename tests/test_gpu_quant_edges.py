"""The quantisers' codes next to a tie and for values without an order, and the dequantisers' wide and narrow
stores: bit for bit against the oracle."""
import numpy as np
import pytest
import torch

from gpu_helpers import dev, host, same_bits
from oracle import synth

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def C():
    from tritiercache_amd import _C
    return _C


def _edges(n, h, d):
    """Values [n, h, d]: N(0, 1) beside groups whose quotients lie on and a few ulps around 0.5, 1.5 and 2.5, and
    groups that hold infinities, NaNs, denormals, equal values, signed zeros and the largest numbers."""
    x = synth.normal(61, 0, (n, h, d)).copy()
    lo, s = np.float32(-1.25), np.float32(0.37)
    near = [(lo + s * np.float32(t)) * (1 + e) for e in (0.0, 1.2e-7, -1.2e-7, 1e-6, -1e-6) for t in (0.5, 1.5, 2.5)]
    row = np.resize(np.array([lo, lo + 3 * s, *near], np.float32), n)
    x[:, 0, : d // 2] = row[:, None]
    x[:, 0, 0], x[0, 0, 1], x[n // 2, 0, 2], x[n - 1, 0, 3] = 0.5, np.nan, np.inf, -np.inf
    x[:, 0, 4] = np.resize(np.array([1e-42, 3e-42, -2e-42, 0.0, -0.0], np.float32), n)
    x[:, 0, 5] = np.resize(np.array([3.4e38, -3.4e38, 1e38], np.float32), n)
    x[:, 0, 6] = np.resize(np.array([2.5e30, -1e30, 1e30], np.float32), n)
    x[1, 0, 7] = np.nan
    # the same along the channels (V groups)
    x[2, 0] = np.resize(np.array([lo, lo + 3 * s, *near], np.float32), d)
    x[3, 0, :] = np.resize(np.array([1e-42, -0.0, 0.0], np.float32), d)
    x[4, 0, d - 1] = np.nan
    x[5, 0, d // 2] = np.inf
    x[6, 0] = np.resize(np.array([3.4e38, -3.4e38, 0.0], np.float32), d)
    return x


@pytest.mark.parametrize("h,d,nb,kgs,fp16", [(1, 16, 1, 16, False), (3, 80, 2, 32, True), (2, 256, 3, 16, False),
                                             (5, 96, 7, 16, True), (1, 1040, 2, 16, False), (3, 18, 3, 16, False)])
@pytest.mark.parametrize("shift", [0, 1])
def test_codes_and_stores_at_the_edges(C, oracle, h, d, nb, kgs, fp16, shift):
    """`shift`: outputs of the dequantisers one float past a 16-byte boundary (the narrow stores)."""
    n, meta = nb * kgs, "fp16" if fp16 else "fp32"
    mdt = torch.uint16 if fp16 else torch.float32
    x = _edges(n, h, d)
    xd = dev(x)
    kp = torch.zeros((nb, kgs // 16, h, d), dtype=torch.int32, device="cuda")
    ks, kz = (torch.zeros((nb, h, d), dtype=mdt, device="cuda") for _ in range(2))
    C.quantize_k_blocks(xd, kp, ks, kz, nb, h, d, kgs, meta)
    want = [oracle.quantize_k(x[b * kgs:(b + 1) * kgs], kgs, fp16) for b in range(nb)]
    p, s, z = (np.stack([w[i] for w in want]) for i in range(3))
    assert same_bits(host(kp).reshape(p.shape), p) and same_bits(host(ks), s) and same_bits(host(kz), z)
    out = torch.zeros(n * h * d + 4, dtype=torch.float32, device="cuda")[shift:shift + n * h * d]
    C.dequantize_k(kp, ks, kz, out, nb, h, d, kgs, meta)
    assert same_bits(host(out).reshape(n, h, d), oracle.dequantize_k(p, s, z, nb, h, d, kgs, fp16))
    if d % 16:
        return
    vp = torch.zeros((n, h, d // 16), dtype=torch.int32, device="cuda")
    vs, vz = (torch.zeros((n, h), dtype=mdt, device="cuda") for _ in range(2))
    C.quantize_v_block(xd, vp, vs, vz, h, d, n, meta)
    p, s, z = oracle.quantize_v(x, fp16)
    assert same_bits(host(vp), p) and same_bits(host(vs), s) and same_bits(host(vz), z)
    out.zero_()
    C.dequantize_v(vp, vs, vz, out, n, h, d, meta)
    assert same_bits(host(out).reshape(n, h, d), oracle.dequantize_v(p, s, z, n, h, d, fp16))


# more than a wave per SIMD, where the quantisers' codes come from the reciprocal and the K stores are wide
@pytest.mark.parametrize("h,d,nb,kgs,fp16", [(1, 16, 4099, 16, False), (3, 80, 277, 32, True), (2, 256, 131, 16, False),
                                             (5, 96, 139, 16, True), (1, 1040, 67, 16, False), (3, 18, 1217, 16, False)])
@pytest.mark.parametrize("shift", [0, 1])
def test_codes_and_stores_at_the_edges_of_large_launches(C, oracle, h, d, nb, kgs, fp16, shift):
    test_codes_and_stores_at_the_edges(C, oracle, h, d, nb, kgs, fp16, shift)


@pytest.mark.parametrize("blocks", [255, 256, 257])
def test_both_sides_of_a_wave_per_simd(C, oracle, blocks):
    """65,536 threads and a block less and more: 2 heads of 128 channels in blocks of 32 (K), V rows of 8 words."""
    test_codes_and_stores_at_the_edges(C, oracle, 2, 128, blocks, 32, True, 0)
