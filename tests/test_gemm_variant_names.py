"""Names of the GEMM variants that the timer records: one per kernel, so that a
report keyed by them keeps every time."""
from remifa_amd import api


def test_fp8_variants_have_their_own_names():
    names = {t: api.gemm_variant_name((3 << 8) | t) for t in (4, 5, 15)}
    assert len(set(names.values())) == 3
    assert names[4].startswith("gemm_fp8_big_kernel<float>") and "256x256 tile" in names[4]
    assert names[5].startswith("gemm_fp8_kernel<float>") and "128x128 tile" in names[5]
    assert names[15].startswith("splitk_reduce_kernel<float>")
    assert "_Float16" in api.gemm_variant_name((3 << 8) | (1 << 4) | 4)


def test_every_variant_has_its_own_name():
    codes = [(k << 8) | (o << 4) | t for k in (0, 1, 2, 4) for o in (0, 1)
             for t in (0, 1, 2, 3, 4, 5, 6, 7, 8)]
    assert len({api.gemm_variant_name(c) for c in codes}) == len(codes)
