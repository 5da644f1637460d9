"""Register-staged GEMM (pe_gemm_rs.h): float16 operands that are not whole
aligned vectors and float32 operands as three bfloat16 terms, at the edges of
tiles, vectors and slabs, in every operand layout, against float64."""
import ctypes

import pytest
import torch

from pto_einsum import abi, einsum, launch

pytestmark = pytest.mark.gpu

EPS = 2.0 ** -24
LAYOUTS = ["bij,bjk->bik", "bij,bkj->bik", "bji,bjk->bik", "bji,bkj->bik"]


def _operands(eq, nb, M, N, K, dtype, seed, off=0):
    d = dict(b=nb, i=M, j=K, k=N)
    g = torch.Generator().manual_seed(seed)
    out = []
    for s in eq.split("->")[0].split(","):
        shape = [d[c] for c in s]
        n = shape[0] * shape[1] * shape[2]
        out.append(torch.randn(n + off, generator=g).to(dtype).cuda()[off:].view(shape))
    return out


def _check(eq, a, b, K):
    """Within K roundings of sum |a||b|, the bound of any order of K fused
    terms, each 2^-24 of a normal result or 2^-150 of a subnormal one, and the
    same bits on a second call.  (Too wide to see an error in the third term:
    test_float32_single_products and test_float32_error_at_edges do.)"""
    got = einsum(eq, a, b)
    want = torch.einsum(eq, a.double(), b.double())
    mag = torch.einsum(eq, a.double().abs(), b.double().abs())
    bad = (got.double() - want).abs() > K * (EPS * mag + 2.0 ** -150)
    assert not bool(bad.any()), (eq, tuple(a.shape), tuple(b.shape), int(bad.sum()))
    assert torch.equal(got, einsum(eq, a, b))


@pytest.mark.parametrize("eq", LAYOUTS)
@pytest.mark.parametrize("nb,M,N,K", [
    (1, 9, 8, 9), (1, 63, 65, 8), (2, 65, 63, 15), (1, 64, 70, 33), (3, 70, 90, 31),       # 64x64 tiles, 32-k slabs
    (20, 201, 99, 65), (1, 300, 200, 64), (1, 700, 129, 71), (40, 129, 131, 127),          # 128x128, 64-k slabs
    (40, 136, 250, 129), (1, 1100, 1300, 193), (1, 1001, 301, 2003),                       # splits
    (2, 2001, 1003, 1000),
])
def test_float16_unaligned_rows(eq, nb, M, N, K):
    a, b = _operands(eq, nb, M, N, K, torch.float16, M + N + K)
    _check(eq, a, b, K)


# Sizes that float32 operands take the kernel at whatever their alignment:
# tiles without much padding, K tails, tiles that end inside a vector, element
# offsets, K splits.
EDGES = [(180, 127, 125, 64, 1), (180, 125, 128, 67, 0), (90, 255, 100, 79, 0), (180, 126, 97, 81, 3),
         (3, 1025, 1023, 101, 0), (180, 128, 127, 192, 0), (90, 128, 252, 193, 2), (3, 1021, 1026, 207, 0),
         (1, 1700, 1800, 777, 0), (1, 767, 765, 4099, 1), (1, 768, 768, 4096, 0)]


@pytest.mark.parametrize("eq", LAYOUTS)
@pytest.mark.parametrize("nb,M,N,K,off", EDGES)
def test_float32_as_bfloat16_terms(eq, nb, M, N, K, off):
    a, b = _operands(eq, nb, M, N, K, torch.float32, M + N + K, off)
    _check(eq, a, b, K)


@pytest.mark.parametrize("eq", LAYOUTS)
@pytest.mark.parametrize("nb,M,N,K,off", EDGES)
def test_float32_single_products(eq, nb, M, N, K, off):
    """Sums with one non-zero product are that product rounded once, but for
    seven roundings of the low accumulator (at most 2^-6.9 of it, so 2^-28.1)
    and the omitted x2 y2 (2^-33), twice that if sums are cut off: 1 + 2^-3
    roundings.  Scaled operands: products whose terms, or which themselves, are
    subnormal (tiles that float32 matrix cores compute again)."""
    a, b = _operands(eq, nb, M, N, K, torch.float32, M + K, off)
    s1 = eq.split("->")[0].split(",")[1]
    kn = b if s1 == "bjk" else b.transpose(1, 2)
    at = (torch.arange(N, device="cuda") * 7 + 3) % K
    pick = torch.zeros(K, N, device="cuda")
    pick[at, torch.arange(N, device="cuda")] = 1.0
    kn.mul_(pick)
    row = a if eq.startswith("bij") else a.transpose(1, 2)
    for scale in (1.0, 2.0 ** -50, 2.0 ** -9, 2.0 ** -7, 2.0 ** -6):    # 2^-50, -59, -66, -72 in all
        a.mul_(scale), b.mul_(scale)
        want = row[:, :, at].double() * kn[:, at, torch.arange(N, device="cuda")].double()[:, None, :]
        got = einsum(eq, a, b).double()
        bad = (got - want).abs() > EPS * (1 + 2.0 ** -3) * want.abs() + 2.0 ** -149
        assert not bool(bad.any()), (scale, int(bad.sum()), float(((got - want) / want).abs().max()))


@pytest.mark.parametrize("eq", LAYOUTS)
@pytest.mark.parametrize("nb,M,N,K,off", EDGES)
def test_float32_error_at_edges(eq, nb, M, N, K, off):
    """The relative error against 64 bits is well below that of float32 matrix
    cores (the explicit 128x128 tile), which round eight times as often; a
    wrong or missing term, or the other kernel, is above the line."""
    a, b = _operands(eq, nb, M, N, K, torch.float32, M + N, off)
    want = torch.einsum(eq, a.double(), b.double())
    ta, tb = not eq.startswith("bij"), eq.split("->")[0].split(",")[1] == "bkj"
    d = launch.GemmDesc(dtype=launch.DT_F32, batch_shape=[nb], a_bstride=[M * K], b_bstride=[K * N], c_bstride=[M * N],
                        M=M, N=N, K=K, a_ms=1 if ta else K, a_ks=M if ta else 1, b_ks=1 if tb else N,
                        b_ns=K if tb else 1, c_ms=N, c_ns=1, a_numel=nb * M * K, b_numel=nb * K * N,
                        c_numel=nb * M * N, split_k=1, tile=128)
    got, ref = einsum(eq, a, b), torch.empty_like(want, dtype=torch.float32)
    st = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    assert abi.bind().pe_gemm(ctypes.byref(abi.gemm_desc(d)), *(ctypes.c_void_p(t.data_ptr()) for t in (a, b, ref)),
                              None, ctypes.c_int64(0), st) == 0
    e = [float((x.double() - want).norm() / want.norm()) for x in (got, ref)]
    assert e[0] <= 0.6 * e[1], e


@pytest.mark.parametrize("eq,layout", [(LAYOUTS[0], (0, 1)), (LAYOUTS[1], (0, 0)), (LAYOUTS[2], (1, 1))])
@pytest.mark.parametrize("nb,M,N,K", [(64, 128, 384, 192), (16, 512, 512, 512), (1, 2048, 1536, 2048)])
def test_float32_error_is_no_larger_than_float32_mfmas(eq, layout, nb, M, N, K):
    """Against 64 bits, next to the same product on float32 matrix cores (the
    explicit 128x128 tile)."""
    a, b = _operands(eq, nb, M, N, K, torch.float32, 11)
    want = torch.einsum(eq, a.double(), b.double())
    got = einsum(eq, a, b)
    d = launch.GemmDesc(dtype=launch.DT_F32, batch_shape=[nb], a_bstride=[M * K], b_bstride=[K * N], c_bstride=[M * N],
                        M=M, N=N, K=K, a_ms=1 if layout[0] else K, a_ks=M if layout[0] else 1,
                        b_ks=N if layout[1] else 1, b_ns=1 if layout[1] else K, c_ms=N, c_ns=1,
                        a_numel=nb * M * K, b_numel=nb * K * N, c_numel=nb * M * N, split_k=1, tile=128)
    ref = torch.empty_like(got)
    st = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    assert abi.bind().pe_gemm(ctypes.byref(abi.gemm_desc(d)), *(ctypes.c_void_p(t.data_ptr()) for t in (a, b, ref)),
                              None, ctypes.c_int64(0), st) == 0
    e = [float((x.double() - want).norm() / want.norm()) for x in (got, ref)]
    assert e[0] <= e[1], e


def test_float32_range():
    """Elements and sums outside the split's range: inf and NaN reach exactly
    the outputs whose sums hold them, tiny and subnormal elements keep their
    float32 accuracy, sums near the largest float32 stay finite."""
    eq, nb, M, N, K = LAYOUTS[0], 60, 127, 383, 200
    a, b = _operands(eq, nb, M, N, K, torch.float32, 5)
    a[3, 7, 11], b[9, 100, 20], a[20, 126, 199] = float("inf"), float("nan"), float("-inf")
    a[30, 5] = 2.0 ** 120
    b[30, :, 6] = 2.0 ** 9     # overflows to inf as float32 does
    got, want = einsum(eq, a, b), torch.einsum(eq, a.double(), b.double())
    big = want.abs() > 3.4028235677973366e38    # halfway past the largest float32
    for f in (torch.isnan, torch.isposinf, torch.isneginf):
        assert torch.equal(f(got) & ~big, f(want) & ~big)
    assert torch.equal(torch.isinf(got)[big], torch.ones_like(got[big], dtype=torch.bool))
    for scale in (2.0 ** -104, 2.0 ** -126, 2.0 ** -140):
        a, b = _operands(eq, nb, M, N, K, torch.float32, 6)
        a[5] *= scale            # one batch wholly tiny, one element of another
        a[7, 64, 3] *= scale
        b[8, 5:50] *= scale
        _check(eq, a, b, K)
    a, b = _operands(eq, nb, M, N, K, torch.float32, 7)
    a[4], b[4] = 2.0 ** 60, 1.9 * 2.0 ** 66 / K     # sums just below 2^127
    a[6], b[6] = 2.0 ** 60, 1.95 * 2.0 ** 67 / K    # ... and above it
    assert bool(torch.isfinite(einsum(eq, a, b)).all())
    _check(eq, a, b, K)


def test_float32_large_elements_and_decays():
    """Elements that the scale takes past the range against small ones, sums
    past it that float32 holds, and elements that decay into subnormals."""
    eq, nb, M, N, K = LAYOUTS[0], 60, 128, 384, 200
    a, b = _operands(eq, nb, M, N, K, torch.float32, 8)
    a[2] *= 2.0 ** 110
    b[2] *= 2.0 ** -100
    a[5, 3, 7], b[5] = 2.0 ** 127, b[5] * 2.0 ** -20
    a[8] *= 2.0 ** 40
    b[8] *= 2.0 ** 45
    a[11:] *= 2.0 ** -torch.arange(K, device="cuda").float()
    _check(eq, a, b, K)
