"""Several right-hand sides: the matrix-core solves and residuals at the edges
of their blocks (128 rows, 16 columns, groups of columns side by side, the
fold from the seventh block row on), and the smallest workspaces."""
import numpy as np
import pytest

import oracle as orc
from helpers import to_dev, to_np

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,nrhs,lu_t", [(1, 2, "f32"), (16, 16, "f16"), (127, 17, "f32"),
                                         (129, 2, "f16"), (300, 64, "f32"), (1025, 33, "f16"),
                                         (1152, 130, "f32")])
@pytest.mark.parametrize("trans", [False, True])
@pytest.mark.parametrize("pad", [0, 3])
def test_getrs_many_columns(handle, gpu, n, nrhs, lu_t, trans, pad):
    """Against the FP64 substitution with the same factors, within the bound
    of the one-column solves (64 n u), and each column as a call with half
    the columns gives it, bit for bit."""
    import torch
    import remifa_amd as rf
    a = orc.gen_diagdom_alpha(n, 3, 1.2) + np.eye(n, dtype=np.float32)
    f = orc.lu_nopiv("rl", orc.cfg(), np.asfortranarray(a), 64)
    raw = orc.f32_to_f16_bits(f) if lu_t == "f16" else f
    f = orc.f16_bits_to_f32(raw) if lu_t == "f16" else f
    dlu = to_dev(raw, gpu, ld=n + pad)
    b = orc.gen_uniform(n, nrhs, 17)
    db = to_dev(b, gpu, ld=n + 1)
    rf.getrs_nopiv(handle, dlu, db, trans=trans)
    k = max(2, nrhs // 2)
    dh = to_dev(np.asfortranarray(b[:, nrhs - k:]), gpu)
    rf.getrs_nopiv(handle, dlu, dh, trans=trans)
    torch.cuda.synchronize()
    x = to_np(db)
    assert np.array_equal(x[:, nrhs - k:].view(np.uint32), to_np(dh).view(np.uint32))
    x64 = orc.getrs_f64(f.astype(np.float64), b.astype(np.float64), trans=trans)
    assert np.abs(x - x64).max() <= 64 * n * 2.0**-24 * np.abs(x64).max()


@pytest.mark.parametrize("n,nrhs,pad", [(1, 2, 0), (31, 16, 1), (255, 17, 0), (257, 40, 3),
                                        (700, 64, 0), (1000, 70, 4)])
def test_residual_many_columns(handle, gpu, n, nrhs, pad):
    """Against the oracle's row-ordered FP64 sum: both within (n + 2) u_64
    (|A||x| + |b|)."""
    import torch
    import remifa_amd as rf
    a = orc.gen_diagdom_alpha(n, 8, 1.05)
    rng = np.random.default_rng(n)
    x = np.asfortranarray(rng.standard_normal((n, nrhs)))
    b = np.asfortranarray(rng.standard_normal((n, nrhs)))
    dr = to_dev(np.zeros((n, nrhs), order="F"), gpu, ld=n + 2)
    rf.residual_f64(handle, to_dev(a, gpu, ld=n + pad), to_dev(x, gpu, ld=n + 1), to_dev(b, gpu),
                    dr)
    torch.cuda.synchronize()
    bound = (n + 2) * 2.0**-53 * (np.abs(a.astype(np.float64)) @ np.abs(x) + np.abs(b))
    assert np.all(np.abs(to_np(dr) - orc.residual_f64(a, x, b)) <= 2 * bound)


@pytest.mark.parametrize("n,nrhs", [(200, 1), (300, 2), (520, 15), (700, 40)])
@pytest.mark.parametrize("trans", [False, True])
def test_refinement_in_small_workspace(gpu, n, nrhs, trans):
    """A caller's workspace that holds one group of 16 columns at a time (the
    sync words, the inverted blocks, 16 tagged columns, the fp32 and FP64
    columns, partials of a few chunks) takes the narrow passes: accepted, and
    as accurate as with the library's own workspace."""
    import torch
    import remifa_amd as rf
    al = lambda v: (v + 255) // 256 * 256
    nb = -(-n // 128)
    solve = 256 + 2 * 4 * 128 * 128 * nb + 8 * n * 16
    nr = min(nrhs, 16)
    part = 8 * nr * n * max(-(-n // 512), -(-n // (2048 if nr == 1 else 256)))
    size = al(solve) + al(4 * n * nrhs) + al(8 * n * nrhs) + al(part) + al(8 * n) + al(
        8 * (2 * nrhs + 2))
    a = orc.gen_diagdom_alpha(n, 21, 1.1)
    lu = to_dev(orc.lu_nopiv("rl", orc.cfg(), a, 64), gpu)
    b = orc.gen_uniform(n, nrhs, 5).astype(np.float64)
    da, db = to_dev(a, gpu), to_dev(np.asfortranarray(b), gpu)
    for ws in (None, torch.empty(size, dtype=torch.uint8, device=gpu)):
        h = rf.Handle()
        if ws is not None:
            h.set_workspace(ws)
        dx = to_dev(np.zeros((n, nrhs), order="F"), gpu)
        it, be, _ = rf.ir_solve(h, da, lu, db, dx, tol=1e-14, maxit=20, trans=trans)
        torch.cuda.synchronize()
        assert it >= 0 and be <= 1e-14
        m = np.asfortranarray(a.T) if trans else a
        assert orc.backward_error(m, b, to_np(dx)) <= 1e-14
