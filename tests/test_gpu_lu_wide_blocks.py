"""Outer blocks wider than the matrix, too wide for the sums inside the slice
kernel, and workspaces without room for its operand copies."""
import numpy as np
import pytest

import oracle as orc
from helpers import assert_parity, to_dev, to_np

pytestmark = pytest.mark.gpu

# (storage, inner, outer, panel precision) as in the slice kernel's test
TUPLES = {"f32": (0, 0, 0, 0), "f32tc": (0, 2, 2, 0), "f16tc": (1, 2, 2, 1), "f16bf": (1, 4, 4, 1),
          "buf32": (1, 0, 2, 0), "buftc": (1, 2, 2, 0), "bufbf": (1, 4, 4, 0)}


def _cfg(rf, name, ib):
    W, I, O, OP = TUPLES[name]
    return rf.api.make_config(W=W, I=I, O=O, OP=OP, ib=ib)


@pytest.mark.parametrize("name,algo", [("f32", "ll"), ("f32tc", "ll"), ("f16tc", "ll"),
                                       ("f32", "rl"), ("f16bf", "rl")])
def test_block_wider_than_matrix(handle, gpu, name, algo):
    """nb far above n is one outer block: the same bits as nb = n, and a
    workspace of the matrix's order (the split-K partials take at most 256
    MiB whatever nb is)."""
    import torch
    import remifa_amd as rf
    n, al = 300, rf.LL if algo == "ll" else rf.RL
    cfg = _cfg(rf, name, 8)
    assert rf.lu_workspace_size(handle, al, cfg, n, n, 10**6) < (256 << 20) + 64 * n * n
    a32 = orc.gen_diagdom_alpha(n, 4, 1.2)
    a = orc.f32_to_f16_bits(a32) if TUPLES[name][0] else a32
    out = []
    for nb in (n, 10**6):
        d = to_dev(a, gpu)
        assert rf.lu_nopiv(handle, d, nb, algo=al, cfg=cfg) == 0
        torch.cuda.synchronize()
        out.append(to_np(d))
    assert np.array_equal(out[0], out[1])


@pytest.mark.parametrize("name,algo,n,nb,pad", [
    ("f32", "rl", 577, 513, 0), ("f32tc", "rl", 600, 600, 1), ("f16tc", "rl", 577, 577, 0),
    ("f16bf", "rl", 600, 520, 2), ("f32", "ll", 1153, 1025, 0), ("buf32", "ll", 1100, 1100, 3)])
def test_wide_blocks_match_oracle(handle, gpu, name, algo, n, nb, pad):
    """The updates between the slices as GEMMs (fp16 storage: ib-wide slices,
    whose rounding points are the oracle's)."""
    import torch
    import remifa_amd as rf
    W, I, O, OP = TUPLES[name]
    a32 = orc.gen_diagdom_alpha(n, 5 + n, 1.2)
    a = orc.f32_to_f16_bits(a32) if W else a32
    d = to_dev(a, gpu, ld=n + pad)
    try:
        handle.set_tuning(32 if OP else 0, 0)
        info = rf.lu_nopiv(handle, d, nb, algo=rf.LL if algo == "ll" else rf.RL,
                           cfg=_cfg(rf, name, 32))
    finally:
        handle.set_tuning(0, 0)
    torch.cuda.synchronize()
    assert info == 0
    oc = {0: orc.F32, 1: orc.F16}
    o = orc.lu_nopiv(algo, orc.LuCfg(oc[W], I, O, oc[OP], oc[OP], oc[OP], oc[OP], 32), a, nb)
    assert_parity(to_np(d), o, f"{name} {algo} n={n} nb={nb}")


@pytest.mark.parametrize("name,n,nb", [("f16bf", 8192, 8192), ("f16tc", 16384, 4096),
                                       ("f32tc", 16384, 4096)])
def test_workspace_without_operand_copies(gpu, name, n, nb):
    """A caller's workspace that holds everything but the operand copies (the
    split-K partials are capped at 256 MiB, the copies take more) is accepted,
    and its factors refine to FP64 accuracy."""
    import torch
    import remifa_amd as rf
    W, _, _, OP = TUPLES[name]
    gen = torch.Generator(device="cuda").manual_seed(7)
    a = (torch.rand((n, n), generator=gen, device=gpu) * 2 - 1).t()
    a.diagonal().copy_(1.1 * a.abs().sum(1))
    b = rf.colmajor_empty(n, 1, dtype=torch.float64)
    b.copy_(torch.rand((n, 1), generator=gen, device=gpu, dtype=torch.float64))
    size = (256 << 20) + (1 << 17)  # partials; the tile slots
    # the fp16 copy, and the second stream's partials
    size += 0 if W else 2 * n * n + (256 << 20)
    h = rf.Handle()
    ws = torch.empty(size, dtype=torch.uint8, device=gpu)
    h.set_workspace(ws)
    cfg = _cfg(rf, name, 8)
    assert rf.lu_workspace_size(h, rf.LL, cfg, n, n, nb) > size
    lu = rf.colmajor_empty(n, n, dtype=torch.float16 if W else torch.float32)
    lu.copy_(a)
    assert rf.lu_nopiv(h, lu, nb, algo=rf.LL, cfg=cfg) == 0
    x = torch.empty_like(b)
    it, be, _ = rf.ir_solve(rf.Handle(), a, lu, b, x, tol=1e-14, maxit=30)
    assert it >= 0 and be <= 1e-14
