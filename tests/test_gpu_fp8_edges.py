"""FP8 operands at the edges of the quantizer's tiles and of the 256 x 256
kernel's tiles, slabs and splits."""
import numpy as np
import pytest

from helpers import to_dev

pytestmark = pytest.mark.gpu


def _reference(x):
    """codes and scale bytes of the rows of x (float32): 2^(floor(log2 amax) -
    8) per 32-block (2^0 if it is zero or not finite), values rounded by
    torch's e4m3 cast after saturation, NaN as sign | 0x7f."""
    import torch
    r, k = x.shape
    kp = -(-k // 32) * 32
    w = np.zeros((r, kp), np.float32)
    w[:, :k] = x
    w = w.reshape(r, kp // 32, 32)
    amax = np.fmax.reduce(np.abs(w), axis=2, initial=0.0)
    ok = (amax > 0) & np.isfinite(amax)
    se = np.where(ok, np.frexp(np.where(ok, amax, 1))[1] - 9, 0)
    with np.errstate(over="ignore"):
        y = np.ldexp(w, -se[:, :, None]).astype(np.float32)
    c = torch.from_numpy(np.clip(np.nan_to_num(y, nan=0.0, posinf=448, neginf=-448), -448, 448))
    c = c.to(torch.float8_e4m3fn).view(torch.uint8).numpy().copy()
    nan = np.isnan(y)
    c[nan] = np.where(np.signbit(y[nan]), 0xFF, 0x7F)
    return c.reshape(r, kp), (se + 127).astype(np.uint8)


@pytest.mark.parametrize("r,k", [(1, 1), (63, 31), (64, 128), (65, 130), (130, 257), (5, 40),
                                 (700, 2050), (3, 4104)])
@pytest.mark.parametrize("rows", [True, False])
@pytest.mark.parametrize("src", ["f16", "f32"])
@pytest.mark.parametrize("pad", [0, 1, 8])
def test_quantizer_edges(handle, gpu, r, k, rows, src, pad):
    """Bit for bit: exponents and codes, every kind of value."""
    import remifa_amd as rf
    rng = np.random.default_rng(r + 5 * k)
    x = (rng.uniform(-1, 1, (r, k)) * np.exp2(rng.integers(-12, 3, (r, k)))).astype(np.float32)
    x[rng.random((r, k)) < 0.05] = 0.0
    x[rng.random((r, k)) < 0.05] = -0.0
    x[rng.random((r, k)) < 0.2] = 17 / 16  # halfway between two codes for most blocks
    flat = x.reshape(-1)
    for i, v in enumerate((np.nan, -np.nan, np.inf, -np.inf)):
        if flat.size > 500:
            flat[(i + 1) * flat.size // 5] = v
    x = x.astype(np.float16).astype(np.float32)
    a = np.asfortranarray(x if rows else x.T)
    host = a.astype(np.float16).view(np.uint16) if src == "f16" else a
    q, s = rf.quantize_fp8(handle, to_dev(np.asfortranarray(host), gpu, ld=a.shape[0] + pad),
                           rows=rows)
    c, se = _reference(x)
    nkb = se.shape[1]
    assert np.array_equal(s.cpu().numpy()[:, :nkb], se)
    assert np.array_equal(q.cpu().numpy()[:, :32 * nkb], c)


@pytest.mark.parametrize("m,n,k,split", [(1, 1, 32, 1), (256, 256, 64, 1), (257, 255, 96, 1),
                                         (300, 700, 1056, 3), (520, 8, 2080, 1),
                                         (255, 513, 256, 1), (768, 256, 224, 1),
                                         (512, 300, 1000, 2)])
@pytest.mark.parametrize("out", ["f32", "f16"])
@pytest.mark.parametrize("beta", [0.0, 1.0])
def test_big_tile_same_bits(handle, gpu, m, n, k, split, out, beta):
    """Both kernels sum the same products in the same order: the same bits,
    and nothing outside C is written."""
    import torch
    import remifa_amd as rf
    g = torch.Generator().manual_seed(m + n + k)
    a = (torch.rand((k, m), generator=g) - 0.5) * torch.exp2(
        torch.randint(-8, 8, (k, m), generator=g).float())
    b = torch.rand((n, k), generator=g) - 0.5
    da, db = a.half().to(gpu), b.half().to(gpu)
    dt = torch.float32 if out == "f32" else torch.float16
    c = torch.rand((n + 1, m + 3), generator=g).to(dt).to(gpu)
    got = []
    handle.set_tuning(split_k=split)
    try:
        for tile in (4, 5):
            handle.set_gemm_tile(tile)
            dc = c.clone()
            rf.gemmex(handle, rf.FP8_TC32, da.t(), db.t(), dc.t()[:m, :n], alpha=-1.0, beta=beta)
            torch.cuda.synchronize()
            got.append(dc)
    finally:
        handle.set_gemm_tile()
        handle.set_tuning()
    assert torch.equal(got[0], got[1])
    assert torch.equal(got[0][:, m:], c[:, m:]) and torch.equal(got[0][n:], c[n:])
    assert not torch.equal(got[0][:n, :m], c[:n, :m])
