"""Outputs of at least 32 MB (where stores are non-temporal) whose rows start on
lines, on halves of lines and off them, through the GEMM kernels, against
float64."""
import pytest
import torch

from pto_einsum import einsum

pytestmark = pytest.mark.gpu

EPS = 2.0 ** -24


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16])
@pytest.mark.parametrize("eq,shapes", [
    ("ij,jk->ik", ((2900, 40), (40, 2944))), ("ij,jk->ik", ((2900, 40), (40, 2928))),
    ("ij,jk->ik", ((2900, 40), (40, 2936))), ("ij,jk->ik", ((2900, 40), (40, 2931))),
    ("ji,jk->ik", ((48, 2904), (48, 2936))),                                      # aligned loads, rows off the lines
    ("ij,jk->ik", ((2999, 257), (257, 3001))), ("ij,kj->ik", ((3000, 512), (3004, 512))),
    ("bshd,bthd->bsht", ((2, 300, 8, 64), (2, 1900, 8, 64))),                     # heads between the rows
    ("bshd,bthd->bsht", ((2, 301, 8, 64), (2, 1901, 8, 64))),
])
def test_rows_on_and_off_lines(eq, shapes, dtype):
    """K roundings of sum |a||b| each."""
    g = torch.Generator().manual_seed(17)
    a, b = (torch.randn(s, generator=g).to(dtype).cuda() for s in shapes)
    K = a.shape[-1] if eq[0:2] != "ji" else a.shape[0]
    got = einsum(eq, a, b)
    assert got.numel() * 4 >= 32 << 20
    want, mag = (torch.einsum(eq, x, y) for x, y in ((a.double(), b.double()), (a.double().abs(), b.double().abs())))
    assert bool(((got.double() - want).abs() <= K * EPS * mag).all())


@pytest.mark.parametrize("eq,shapes", [
    ("ij,jk->ik", ((8200, 32), (32, 8192))), ("ij,kj->ik", ((8200, 520), (8192, 520))),       # short and long K
    ("bhsd,bhtd->bhst", ((1, 17, 2048, 64), (1, 17, 2048, 64))),
])
def test_outputs_beyond_the_last_level_cache(eq, shapes):
    """At least 256 MB: either scope of non-temporal store."""
    test_rows_on_and_off_lines(eq, shapes, torch.float16)
