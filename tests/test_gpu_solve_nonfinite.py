"""Right-hand sides with infinities and NaN: the solve of several columns
propagates them as the solve of one column does, and its other columns do not
notice."""
import numpy as np
import pytest

import oracle as orc
from helpers import to_dev, to_np

pytestmark = pytest.mark.gpu


def _classes(x):
    return np.where(np.isnan(x), 3, np.where(np.isposinf(x), 1, np.where(np.isneginf(x), 2, 0)))


# one row, a last block of one row, blocks with and without the fold; the row
# of the non-finite entry
@pytest.mark.parametrize("n,row", [(1, 0), (129, 128), (300, 0), (300, 299), (1000, 130)])
@pytest.mark.parametrize("nrhs", [2, 20])
@pytest.mark.parametrize("trans", [False, True])
def test_nonfinite_columns(handle, gpu, n, row, nrhs, trans):
    import torch
    import remifa_amd as rf
    a = orc.gen_diagdom_alpha(n, 3, 1.2) + np.eye(n, dtype=np.float32)
    dlu = to_dev(orc.lu_nopiv("rl", orc.cfg(), np.asfortranarray(a), 64), gpu)
    good = orc.gen_uniform(n, nrhs, 17)
    bad = good.copy(order="F")
    values = {0: np.inf, nrhs // 2: -np.inf, nrhs - 1: np.nan}
    for k, v in values.items():
        bad[row, k] = v
    dg, db = to_dev(good, gpu), to_dev(bad, gpu)
    rf.getrs_nopiv(handle, dlu, dg, trans=trans)
    rf.getrs_nopiv(handle, dlu, db, trans=trans)
    torch.cuda.synchronize()
    g, x = to_np(dg), to_np(db)
    for k in range(nrhs):
        if k not in values:
            assert np.array_equal(x[:, k].view(np.uint32), g[:, k].view(np.uint32))
            continue
        one = to_dev(np.asfortranarray(bad[:, k:k + 1]), gpu)
        rf.getrs_nopiv(handle, dlu, one, trans=trans)
        torch.cuda.synchronize()
        assert np.array_equal(_classes(x[:, k]), _classes(to_np(one)[:, 0]))
        if n == 1:
            assert np.array_equal(_classes(x[:, k]), _classes(np.float32([values[k]])))
