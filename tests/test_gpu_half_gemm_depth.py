"""fp16-accumulated products where the register ring's slabs of 16 k-values and
their groups of eight end, with and without the C term, rows and columns at the
edges of a row pair and a wavefront's columns."""
import numpy as np
import pytest

import oracle as orc
from helpers import to_dev, to_np

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("k", [1, 7, 8, 9, 15, 16, 17, 24, 31, 32, 33, 47, 48, 49, 95, 96, 97])
@pytest.mark.parametrize("m,n", [(3, 5), (130, 17), (2177, 513)])
@pytest.mark.parametrize("beta", [0.0, 1.0])
def test_half_sums_depth(handle, gpu, m, n, k, beta):
    import torch
    import remifa_amd as rf
    rng = np.random.default_rng(m + 7 * n + k)
    a = orc.round_to(orc.F16, rng.uniform(-0.25, 0.25, (m, k)).astype(np.float32))
    b = orc.round_to(orc.F16, rng.uniform(-0.25, 0.25, (k, n)).astype(np.float32))
    c = orc.round_to(orc.F16, rng.uniform(-1, 1, (m, n)).astype(np.float32))
    da = to_dev(orc.f32_to_f16_bits(a), gpu, ld=m + 1)
    db = to_dev(orc.f32_to_f16_bits(b), gpu)
    if beta == 0.0:
        dc = to_dev(orc.f32_to_f16_bits(np.full_like(c, np.nan)), gpu, ld=m + 3)
        c = np.zeros_like(c)
    else:
        dc = to_dev(orc.f32_to_f16_bits(c), gpu, ld=m + 3)
    rf.gemmex(handle, rf.TC16, da, db, dc, alpha=-1.0, beta=beta)
    torch.cuda.synchronize()
    ref = orc.f32_to_f16_bits(orc.gemm_sub(orc.FP16, a, b, c, orc.F16))
    got = to_np(dc)
    if beta == 0.0:  # (0 - 0 and -0 differ in sign only)
        got, ref = orc.f16_bits_to_f32(got), orc.f16_bits_to_f32(ref)
    assert np.array_equal(got, ref)
