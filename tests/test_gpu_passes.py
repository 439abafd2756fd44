"""Memory-bound passes (conversions, equilibration) at the edges of their
vectors and workgroups: sizes around 4 / 8 rows and 4 / 8 columns, few rows,
many columns, leading dimensions of every alignment."""
import numpy as np
import pytest

from helpers import to_dev, to_np

pytestmark = pytest.mark.gpu

SHAPES = [(1, 1, 0), (7, 5, 1), (8, 4, 0), (9, 3, 2), (63, 130, 1), (260, 1030, 3),
          (1023, 9, 0), (4099, 37, 1), (2, 70001, 0)]


@pytest.mark.parametrize("m,n,pad", SHAPES)
@pytest.mark.parametrize("src,dst", [("float32", "float16"), ("float16", "float32"),
                                     ("float64", "float16"), ("float16", "bfloat16")])
def test_convert_edges(handle, gpu, m, n, pad, src, dst):
    """One rounding, torch's; nothing outside the block is written."""
    import torch
    import remifa_amd as rf
    s, d = getattr(torch, src), getattr(torch, dst)
    g = torch.Generator().manual_seed(m + n)
    x = torch.randn((n, m), generator=g).to(s).to(gpu)
    a = rf.colmajor_empty(m, n, dtype=s, device=gpu, ld=m + pad)
    a.copy_(x.t())
    buf = torch.full((n + 1, m + pad + 1), 7.0, device=gpu).to(d)
    rf.convert(handle, a, buf.t()[:m, :n])
    torch.cuda.synchronize()
    assert torch.equal(buf[:n, :m], x.to(d))
    assert (buf[:, m:] == 7).all() and (buf[n:] == 7).all()


@pytest.mark.parametrize("m,n,pad", SHAPES)
def test_equilibration_edges(handle, gpu, m, n, pad):
    """Powers of two, so every scale and every scaled entry is exact: r =
    2^-trunc(log2 max), the scaled matrix equal to numpy's products."""
    import torch
    import remifa_amd as rf
    rng = np.random.default_rng(m * 31 + n)
    a = rng.uniform(0.5, 1.0, (m, n)) * np.exp2(rng.integers(-9, 10, (m, 1)) +
                                                rng.integers(-9, 10, (1, n)))
    a = np.asfortranarray((a * rng.choice([-1.0, 1.0], (m, n))).astype(np.float32))
    da = to_dev(a, gpu, ld=m + pad)
    r = torch.zeros(m, device=gpu)
    c = torch.zeros(n, device=gpu)
    q = rf.geequb(handle, da, r, c)

    def trunc2(x):
        return np.exp2(np.trunc(np.log2(x.astype(np.float64))))
    rp = trunc2(np.abs(a).max(1))
    cp = trunc2((np.abs(a) / rp[:, None]).max(0))
    assert q["info"] == 0 and q["amax"] == rp.max()
    assert q["rowcnd"] == rp.min() / rp.max() and q["colcnd"] == cp.min() / cp.max()
    assert np.array_equal(r.cpu().numpy(), 1 / rp) and np.array_equal(c.cpu().numpy(), 1 / cp)
    rf.laqge(handle, da, r, c, 0.01, 0.01, q["amax"])  # both scalings
    torch.cuda.synchronize()
    assert np.array_equal(to_np(da), (a / rp[:, None] / cp[None, :]).astype(np.float32))
