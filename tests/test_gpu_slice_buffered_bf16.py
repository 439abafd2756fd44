"""Left-looking factorization of fp16 storage in fp32 buffers with bf16 inner
updates: the update GEMMs between the slices read the fp16 mirror, both of a
slice in one launch where they take the narrow tiles without split-K."""
import numpy as np
import pytest

import oracle as orc
from helpers import factor_distance, to_dev, to_np

pytestmark = pytest.mark.gpu


# outer update TC32 and BF16; ib-wide and 64-wide slices; split-K forced, which
# takes the two launches. The oracle rounds the fp32 factors to bf16, not their
# fp16 mirror, and 64-wide slices form their own block sums from fp16 operands:
# as close to the FP64 factors as the oracle's.
@pytest.mark.parametrize("outer", [2, 4])
@pytest.mark.parametrize("n,nb,ld_pad,ib,pw,split", [
    (129, 128, 0, 8, 8, 0), (333, 200, 3, 16, 16, 0), (700, 256, 1, 32, 32, 0),
    (600, 256, 8, 8, 8, 2), (129, 128, 1, 8, 0, 0), (577, 200, 3, 16, 0, 0),
    (700, 256, 0, 32, 0, 3)])
def test_buffered_bf16(handle, gpu, outer, n, nb, ld_pad, ib, pw, split):
    import torch
    import remifa_amd as rf
    a32 = orc.gen_diagdom_alpha(n, 5 + n, 1.2)
    a = orc.f32_to_f16_bits(a32)
    d = to_dev(a, gpu, ld=n + ld_pad)
    cfg = rf.api.make_config(W=1, I=4, O=outer, OP=0, ib=ib)
    try:
        handle.set_tuning(pw, split)
        info = rf.lu_nopiv(handle, d, nb, algo=rf.LL, cfg=cfg)
    finally:
        handle.set_tuning(0, 0)
    torch.cuda.synchronize()
    assert info == 0
    g = to_np(d)
    o = orc.lu_nopiv("ll", orc.LuCfg(orc.F16, 4, outer, orc.F32, orc.F32, orc.F32, orc.F32, ib), a,
                     nb)
    f64 = orc.lu_f64(orc.round_to(orc.F16, a32))
    e_o = factor_distance(orc.f16_bits_to_f32(o), f64)
    assert factor_distance(orc.f16_bits_to_f32(g), f64) <= 8 * max(e_o, 2.0**-11)
