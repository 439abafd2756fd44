"""The batched solve where its steps, threads and rows per thread end."""
import numpy as np
import pytest

import oracle as orc
from test_gpu_batched import _batch, _pack

pytestmark = pytest.mark.gpu


# largest order given by the caller: 64 threads, 256 with one row each, with
# two; and one below the orders there are (each is still solved)
@pytest.mark.parametrize("sizes,max_n", [([1, 2, 31, 32, 33, 63, 64], 64),
                                         ([65, 255, 256, 257, 287, 288], 288),
                                         ([1, 289, 320, 321, 511, 512], 512),
                                         ([97, 300, 512], 64), ([289, 512], 256)])
@pytest.mark.parametrize("pad", [0, 1])
def test_batched_solve_edges(handle, gpu, sizes, max_n, pad):
    """Against the FP64 substitution with the same factors, within the bound
    of the other solves, 64 n u; neighbouring right-hand sides stay."""
    import torch
    import remifa_amd as rf
    facs = [orc.lu_nopiv("rl", orc.cfg(), a + np.eye(a.shape[0], dtype=np.float32), 32)
            for a in _batch(sizes, 40)]
    buf, ptrs, n_t, ld_t, _, _ = _pack([np.asfortranarray(f) for f in facs], gpu, pad=pad)
    rng = np.random.default_rng(max_n)
    bs = [rng.uniform(-1, 1, (f.shape[0], 1)).astype(np.float32) for f in facs]
    x = torch.full((sum(sizes) + len(sizes),), 5.0)
    offs = np.cumsum([0] + [n + 1 for n in sizes])
    for b, o in zip(bs, offs):
        x[o:o + b.size] = torch.from_numpy(b[:, 0])
    x = x.to(gpu)
    bptrs = torch.tensor([x.data_ptr() + 4 * int(o) for o in offs[:-1]], dtype=torch.int64,
                         device=gpu)
    rf.getrs_nopiv_batched(handle, n_t, ld_t, ptrs, bptrs, max_n)
    torch.cuda.synchronize()
    got = x.cpu().numpy()
    for f, b, o in zip(facs, bs, offs):
        n = b.size
        want = orc.getrs_f64(f.astype(np.float64), b.astype(np.float64))[:, 0]
        assert np.abs(got[o:o + n] - want).max() <= 64 * n * 2.0**-24 * np.abs(want).max()
        assert got[o + n] == 5.0
