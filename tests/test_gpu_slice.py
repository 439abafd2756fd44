"""The slice kernel of the inner factorization (slice.hpp) at the sizes where
its tiles, units and panels end, for every arithmetic, ib and looking
direction, against the oracle: the entrywise rule of helpers.py (fp16 storage
>= 99.9% identical bits; fp32 storage r_99.9 <= 256), and the pivots outside
the fast reciprocal's range."""
import numpy as np
import pytest

import oracle as orc
from helpers import assert_parity, factor_distance, to_dev, to_np

pytestmark = pytest.mark.gpu


def _lu(handle, gpu, a, algo, nb, pw, ld_pad, kw):
    import torch
    import remifa_amd as rf
    cfg = rf.api.make_config(**kw)
    d = to_dev(a, gpu, ld=a.shape[0] + ld_pad)
    try:
        handle.set_tuning(pw, 0)
        info = rf.lu_nopiv(handle, d, nb, algo=algo, cfg=cfg)
    finally:
        handle.set_tuning(0, 0)
    torch.cuda.synchronize()
    return to_np(d), info


# (storage, inner, outer, panel precision): fp32; fp16 operands on fp32; fp16
# panels with fp16 operands, fp16 sums, bf16 operands; fp32 buffers of fp16
# storage with fp32, fp16 and bf16 inner operands
TUPLES = {"f32": (0, 0, 0, 0), "f32tc": (0, 2, 2, 0), "f16tc": (1, 2, 2, 1), "f16h": (1, 3, 3, 1),
          "f16bf": (1, 4, 4, 1), "buf32": (1, 0, 2, 0), "buftc": (1, 2, 2, 0)}


@pytest.mark.parametrize("name,algo", [(t, a) for t in TUPLES for a in ("ll", "rl")
                                       if not (a == "rl" and t.startswith("buf"))])
@pytest.mark.parametrize("n,nb,pw,ld_pad,ib", [
    (1, 64, 0, 0, 8), (9, 64, 0, 1, 8), (63, 64, 0, 0, 16), (65, 64, 0, 0, 32),
    (129, 200, 0, 3, 8), (130, 128, 8, 0, 8), (191, 128, 0, 0, 64), (333, 200, 32, 2, 16),
    (700, 256, 0, 4, 8)])
def test_slice_edges_match_oracle(handle, gpu, name, algo, n, nb, pw, ld_pad, ib):
    import remifa_amd as rf
    W, I, O, OP = TUPLES[name]
    if name == "f16h" or (algo == "rl" and W):
        # fp16 rounds the sums once per slice where the reference does once
        # per ib block: the same points only with ib-wide slices
        pw = ib
    a32 = orc.gen_diagdom_alpha(n, 5 + n, 1.2)
    a = orc.f32_to_f16_bits(a32) if W else a32
    g, info = _lu(handle, gpu, a, rf.LL if algo == "ll" else rf.RL, nb, pw, ld_pad,
                  dict(W=W, I=I, O=O, OP=OP, ib=ib))
    assert info == (1 if n == 1 else 0)  # (the 1 x 1 matrix of the generator is zero)
    oc = {0: orc.F32, 1: orc.F16}
    c = orc.LuCfg(oc[W], I, O, oc[OP], oc[OP], oc[OP], oc[OP], min(ib, 32))
    o = orc.lu_nopiv(algo, c, a, nb)
    if ib <= 32:
        assert_parity(g, o, f"{name} {algo} n={n} nb={nb} pw={pw} ib={ib}")
        return
    # the oracle takes ib <= 32: as close to the FP64 factors as its ib = 32
    val = (lambda x: orc.f16_bits_to_f32(x)) if W else (lambda x: x)
    f64 = orc.lu_f64(orc.round_to(orc.F16, a32) if W else a32)
    e_o, e_g = factor_distance(val(o), f64), factor_distance(val(g), f64)
    assert e_g <= 8 * max(e_o, 2.0**-11 if W else 2.0**-24)


@pytest.mark.parametrize("scale", [2.0**118, 2.0**-100])
def test_slice_extreme_pivots(handle, gpu, scale):
    """Power-of-two scaling of A scales U and leaves L: with pivots whose
    reciprocals are denormal (2^118 x ~2^7), the exact division takes over.
    L within 4 rounding errors of the unscaled factors' (denormal reciprocals
    have fewer digits: 2^-149 / 2^-126 = 2^-23 relative), U likewise."""
    import remifa_amd as rf
    n = 150
    a = orc.gen_diagdom_alpha(n, 3, 1.2)
    kw = dict(W=0, I=0, O=0, OP=0, ib=8)
    g, i0 = _lu(handle, gpu, a, rf.LL, 256, 0, 0, kw)
    s, i1 = _lu(handle, gpu, (a * np.float32(scale)).astype(np.float32, order="F"), rf.LL, 256, 0,
                0, kw)
    assert i0 == 0 and i1 == 0 and np.isfinite(s).all()
    low = np.tril(np.ones((n, n), bool), -1)
    want = np.where(low, g.astype(np.float64), g.astype(np.float64) * scale)
    size = np.where(low, np.abs(g).max(where=low, initial=0.0), np.abs(g).max() * scale)
    assert (np.abs(s - want) <= 4 * 2.0**-22 * size).all()


@pytest.mark.parametrize("name", ["f32", "f16tc", "f16h"])
@pytest.mark.parametrize("bad", [0, 7, 64, 130])
def test_slice_reports_first_zero_pivot(handle, gpu, name, bad):
    """A zero pivot (its row and column zeroed) is reported 1-based; the
    factors of the columns before it are those of the leading block."""
    import remifa_amd as rf
    W, I, O, OP = TUPLES[name]
    n = 200
    a32 = orc.gen_diagdom_alpha(n, 9, 1.2)
    a32[bad, :] = 0
    a32[:, bad] = 0
    a = orc.f32_to_f16_bits(a32) if W else a32
    kw = dict(W=W, I=I, O=O, OP=OP, ib=8)
    g, info = _lu(handle, gpu, a, rf.LL, 128, 0, 0, kw)
    assert info == bad + 1
    if bad:
        h, _ = _lu(handle, gpu, np.asfortranarray(a[:bad, :bad]), rf.LL, 128, 0, 0, kw)
        assert_parity(g[:bad, :bad], h, f"{name} leading block {bad}")
