"""Equilibration of more columns than a grid has workgroups along them."""
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m", [1, 3])
def test_geequb_wide(handle, gpu, m):
    """65535 chunks of 128 columns and a bit: the row maxima see the first and
    the last column of the range, and every column its own maximum."""
    import torch
    import remifa_amd as rf
    n = 65535 * 128 + 130
    a = rf.colmajor_empty(m, n, dtype=torch.float32)
    a.fill_(0.5)
    a[m - 1, n - 1] = 64.0
    a[0, 7] = 8.0 if m > 1 else 0.25
    r, c = torch.empty(m, device=gpu), torch.empty(n, device=gpu)
    q = rf.geequb(handle, a, r, c)
    big = [0.5] * m  # row maxima, powers of two
    big[0] = 8.0 if m > 1 else 0.5
    big[m - 1] = 64.0
    assert q["info"] == 0 and q["amax"] == 64.0
    rr = torch.tensor([1 / v for v in big], device=gpu)
    assert torch.equal(r, rr)
    # c_j = 1 / max_i |a_ij| r_i, all powers of two
    assert torch.equal(c, 1 / (a * rr[:, None]).amax(0))
    assert q["rowcnd"] == min(big) / max(big)
