"""The residual of several columns in the smallest workspace that a caller may
give it."""
import numpy as np
import pytest

import oracle as orc
from helpers import to_dev, to_np

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,nrhs", [(2, 2), (255, 3), (300, 16), (700, 17), (1025, 40)])
def test_residual_in_small_workspace(gpu, n, nrhs):
    """Partials of 16 columns in chunks of 256: A is read once per 16 columns,
    and the result is the oracle's within (n + 2) u_64 (|A||x| + |b|) each."""
    import torch
    import remifa_amd as rf
    h = rf.Handle()
    ws = torch.empty(8 * min(nrhs, 16) * n * -(-n // 256), dtype=torch.uint8, device=gpu)
    h.set_workspace(ws)
    a = orc.gen_diagdom_alpha(n, 8, 1.05)
    rng = np.random.default_rng(n)
    x = np.asfortranarray(rng.standard_normal((n, nrhs)))
    b = np.asfortranarray(rng.standard_normal((n, nrhs)))
    dr = to_dev(np.zeros((n, nrhs), order="F"), gpu)
    h.timing()
    rf.residual_f64(h, to_dev(a, gpu), to_dev(x, gpu), to_dev(b, gpu), dr)
    torch.cuda.synchronize()
    _, _, work = h.timing_query(4)
    assert work == 4.0 * n * n * -(-nrhs // 16)
    bound = (n + 2) * 2.0**-53 * (np.abs(a.astype(np.float64)) @ np.abs(x) + np.abs(b))
    assert np.all(np.abs(to_np(dr) - orc.residual_f64(a, x, b)) <= 2 * bound)
