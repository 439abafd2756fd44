"""Update GEMM kernels where their tiles, slabs and dispatch rules end."""
import numpy as np
import pytest

import oracle as orc
from helpers import to_dev, to_np

pytestmark = pytest.mark.gpu


# rows around the 128 of a wavefront, columns around the 16 / 32 / 64 of a
# workgroup (the widest needs many tiles), K around the 32-deep slab, odd
# leading dimensions
@pytest.mark.parametrize("m,n,k,pad", [(1, 65, 33, 0), (2, 16, 31, 1), (127, 17, 32, 0),
                                       (128, 64, 64, 3), (129, 33, 95, 1), (255, 15, 1, 2),
                                       (2049, 515, 40, 1), (4100, 1030, 33, 0)])
def test_half_sums_bitexact(handle, gpu, m, n, k, pad):
    """fp16-accumulated products round as the oracle's k-ordered fp16 fma
    chain, bit for bit, at every remainder."""
    import torch
    import remifa_amd as rf
    rng = np.random.default_rng(m + 7 * n + k)
    a = orc.round_to(orc.F16, rng.uniform(-0.25, 0.25, (m, k)).astype(np.float32))
    b = orc.round_to(orc.F16, rng.uniform(-0.25, 0.25, (k, n)).astype(np.float32))
    c = orc.round_to(orc.F16, rng.uniform(-1, 1, (m, n)).astype(np.float32))
    da = to_dev(orc.f32_to_f16_bits(a), gpu, ld=m + pad)
    db = to_dev(orc.f32_to_f16_bits(b), gpu, ld=k + pad)
    dc = to_dev(orc.f32_to_f16_bits(c), gpu, ld=m + pad)
    rf.gemmex(handle, rf.TC16, da, db, dc)
    torch.cuda.synchronize()
    ref = orc.f32_to_f16_bits(orc.gemm_sub(orc.FP16, a, b, c, orc.F16))
    assert np.array_equal(to_np(dc), ref)
