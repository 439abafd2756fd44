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


# one tile and a bit in each direction, the smallest, a single column, K of a
# short slab, below the four stages, around them, and split
@pytest.mark.parametrize("m,n,k,split", [(8, 1, 8, 1), (264, 255, 40, 1), (248, 257, 24, 1),
                                         (520, 3, 136, 1), (256, 512, 128, 1),
                                         (1000, 700, 2008, 1), (272, 300, 1000, 3),
                                         (8, 600, 200, 2)])
@pytest.mark.parametrize("out", ["f32", "f16"])
@pytest.mark.parametrize("beta", [0.0, 1.0])
def test_big_tile_edges(handle, gpu, m, n, k, split, out, beta):
    """The 256 x 256 kernel on partial tiles and slabs: within 2 (k + 2) u
    (|A||B| + |C|) of the FP64 product (any summation order), plus one
    rounding of an fp16 result, and nothing outside C is touched. What lies
    beside the operands is NaN and must not reach the result."""
    import torch
    import remifa_amd as rf
    g = torch.Generator().manual_seed(m + 3 * n + k)
    nan = float("nan")
    ab = torch.full((k, m + 8), nan, dtype=torch.float16)
    ab[:, :m] = (torch.rand((k, m), generator=g) - 0.5).half()
    bb = torch.full((n, k + 16), nan, dtype=torch.float16)
    bb[:, :k] = (torch.rand((n, k), generator=g) - 0.5).half()
    dt = torch.float32 if out == "f32" else torch.float16
    cb = torch.full((n + 2, m + 3), 9.0, dtype=dt)
    cb[:n, :m] = (torch.rand((n, m), generator=g) - 0.5).to(dt)
    da, db, dc = ab.to(gpu), bb.to(gpu), cb.to(gpu)
    handle.set_gemm_tile(4)
    handle.set_tuning(split_k=split)
    try:
        rf.gemmex(handle, rf.TC32, da.t()[:m], db.t()[:k], dc.t()[:m, :n], alpha=-1.0, beta=beta)
        torch.cuda.synchronize()
    finally:
        handle.set_gemm_tile()
        handle.set_tuning()
    a, b, c = ab[:, :m].double().t(), bb[:, :k].double().t(), cb[:n, :m].double().t()
    ref = beta * c - a @ b
    mag = a.abs() @ b.abs() + beta * c.abs()
    got = dc.cpu()
    tol = 2 * (k + 2) * 2.0**-24 * mag
    if out == "f16":
        tol = tol + 2.0**-11 * ref.abs() + 2.0**-24
    assert ((got[:n, :m].double().t() - ref).abs() <= tol).all()
    assert (got[:, m:] == 9).all() and (got[n:] == 9).all()


# element-aligned operands: rows and K around the 8 (4) of a chunk, the tiles'
# edges, K around a slab, a leading dimension below a chunk, split
@pytest.mark.parametrize("m,n,k,pad,split", [(1, 1, 1, 0, 1), (3, 5, 200, 0, 1), (9, 31, 64, 1, 1),
                                             (33, 257, 63, 3, 1), (129, 127, 129, 0, 1),
                                             (255, 33, 128, 1, 1), (257, 130, 1000, 2, 3),
                                             (301, 299, 256, 1, 1)])
@pytest.mark.parametrize("ctype", ["TC32", "BF16_TC32", "FP32"])
@pytest.mark.parametrize("tile", [0, 1, 5])
def test_unaligned_operands(handle, gpu, m, n, k, pad, split, ctype, tile):
    """Within 2 (k + 2) u (|A||B| + |C|) of the FP64 product of the rounded
    operands; the padding is NaN and must not reach the result. The operands
    start at an odd element."""
    import torch
    import remifa_amd as rf
    g = torch.Generator().manual_seed(m + 3 * n + k)
    dt = torch.float32 if ctype == "FP32" else torch.float16

    def operand(r, c):  # r x c column-major, ld r + pad, NaN beside it
        buf = torch.full((1 + c * (r + pad),), float("nan"), dtype=dt)
        v = buf[1:].view(c, r + pad).t()[:r]
        v.copy_((torch.rand((r, c), generator=g) - 0.5).to(dt))
        return v.double(), buf.to(gpu)[1:].view(c, r + pad).t()[:r]
    a, da = operand(m, k)
    b, db = operand(k, n)
    if ctype == "BF16_TC32":
        a, b = a.bfloat16().double(), b.bfloat16().double()
    c = torch.rand((n, m + 1), generator=g) - 0.5
    dc = c.to(gpu)
    handle.set_gemm_tile(tile)
    handle.set_tuning(split_k=split)
    try:
        rf.gemmex(handle, getattr(rf, ctype), da, db, dc.t()[:m], alpha=-1.0, beta=1.0)
        torch.cuda.synchronize()
    finally:
        handle.set_gemm_tile()
        handle.set_tuning()
    c64 = c[:, :m].double().t()
    tol = 2 * (k + 2) * 2.0**-24 * (a.abs() @ b.abs() + c64.abs())
    assert ((dc.cpu()[:, :m].double().t() - (c64 - a @ b)).abs() <= tol).all()
    assert torch.equal(dc.cpu()[:, m:], c[:, m:])
