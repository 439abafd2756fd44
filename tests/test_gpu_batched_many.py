"""The two instantiations of the batched factorization give the same bits: a
batch too large for one workgroup per matrix against one of few."""
import pytest

from test_gpu_batched import _batch, _pack

pytestmark = pytest.mark.gpu


# sizes of a bucket (its ends among them), repeated beyond the batch length
# from which the other instantiation runs; the smallest bucket has only one
@pytest.mark.parametrize("sizes,repeat", [([64, 33, 1, 32], 700), ([128, 65, 97, 96], 300),
                                          ([256, 129, 161, 250], 150), ([512, 257, 289], 270)])
@pytest.mark.parametrize("ctype", ["TC32", "BF16_TC32"])
def test_many_as_few(handle, gpu, sizes, repeat, ctype):
    import torch
    import remifa_amd as rf
    ct = getattr(rf, ctype)
    mats = _batch(sizes, 60)
    buf, ptrs, n_t, ld_t, offs, _ = _pack(mats, gpu)
    many = buf.repeat(repeat)
    mptr = torch.tensor([many.data_ptr() + 4 * (r * buf.numel() + int(o))
                         for o in offs for r in range(repeat)], dtype=torch.int64, device=gpu)
    info = torch.full((len(sizes),), -7, dtype=torch.int32, device=gpu)
    rf.lu_nopiv_batched(handle, ct, n_t, ld_t, ptrs, info, max(sizes))
    minfo = torch.full((len(sizes) * repeat,), -7, dtype=torch.int32, device=gpu)
    rf.lu_nopiv_batched(handle, ct, n_t.repeat_interleave(repeat), ld_t.repeat_interleave(repeat),
                        mptr, minfo, max(sizes))
    torch.cuda.synchronize()
    assert torch.equal(minfo, info.repeat_interleave(repeat))
    assert torch.equal(many.view(repeat, -1).view(torch.int32),
                       buf.view(torch.int32).expand(repeat, -1))
