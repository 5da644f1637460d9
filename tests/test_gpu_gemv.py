"""Matrix-vector contractions (pe_gemv.hip): M or N of 1, W contiguous along k
(rows) or along n (columns), at the sizes where the kernels change: lanes per
row, rows per wave, one x per row, K splits and their two reductions, K tails,
partial tiles, unaligned rows and bases, strided outputs and batches."""
import ctypes

import pytest
import torch

from pto_einsum import abi, einsum, launch

pytestmark = pytest.mark.gpu

EPS = 2.0 ** -24


def _check(eq, a, b):
    """Every output within K roundings of sum |a||b| (any summation order of K
    fused terms), and the same bits on a second call."""
    got = einsum(eq, a, b)
    want = torch.einsum(eq, a.double(), b.double())
    mag = torch.einsum(eq, a.double().abs(), b.double().abs())
    s0, s1 = eq.split("->")[0].split(",")
    size = dict(zip(s0, a.shape)) | dict(zip(s1, b.shape))
    K = 1
    for c in set(s0) & set(s1) - set(eq.split("->")[1]):
        K *= size[c]
    assert got.shape == want.shape and got.dtype == torch.float32
    assert bool(((got.double() - want).abs() <= K * EPS * mag + 1e-44).all()), (eq, tuple(a.shape), tuple(b.shape))
    assert torch.equal(got, einsum(eq, a, b))


def _rand(shape, dtype, seed, off=0):
    """Contiguous tensor whose base is `off` elements past an aligned one."""
    g = torch.Generator().manual_seed(seed)
    n = 1
    for s in shape:
        n *= s
    return torch.randn(n + off, generator=g).to(dtype).cuda()[off:].view(shape)


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16])
@pytest.mark.parametrize("eq,s0,s1", [
    ("ij,j->i", (70, 8), (8,)),               # 4 lanes a row, K of one or two vectors
    ("ij,j->i", (1, 4099), (4099,)),          # a dot product by another name
    ("ij,j->i", (513, 77), (77,)),            # K tail, odd row pitch
    ("ij,j->i", (1000, 96), (96,)),
    ("ij,j->i", (300, 250), (250,)),
    ("ij,j->i", (257, 1000), (1000,)),
    ("ij,j->i", (8200, 4100), (4100,)),       # one row for 64 lanes, U vectors of it in flight
    ("ij,j->i", (5, 70001), (70001,)),        # K split, wave reduction, odd pitch
    ("ij,j->i", (40, 40000), (40000,)),       # K split, ordered reduction
    ("i,ij->j", (9,), (9, 8)),
    ("i,ij->j", (1000,), (1000, 9)),          # overlapping last vector, K split
    ("i,ij->j", (777,), (777, 513)),
    ("i,ij->j", (4096,), (4096, 1000)),
    ("i,ij->j", (30000,), (30000, 64)),
    ("i,ij->j", (64,), (64, 16384)),
    ("i,i->", (1000,), (1000,)),
    ("i,i->", (1 << 20,), (1 << 20,)),
    ("i,i->", (999999,), (999999,)),
    ("bi,bi->b", (3, 40), (3, 40)),           # one x per row
    ("bi,bi->b", (1001, 77), (1001, 77)),
    ("bi,bi->b", (9000, 1030), (9000, 1030)),
    ("bi,bni->bn", (37, 60), (37, 5, 60)),    # fewer rows per batch than a tile
    ("bni,bi->nb", (4, 300, 24), (4, 24)),    # strided output
    ("bhd,bthd->bht", (2, 3, 64), (2, 301, 3, 64)),
    ("bhd,bthd->bht", (2, 3, 72), (2, 130, 3, 72)),
    ("bht,bthd->bhd", (2, 3, 301), (2, 301, 3, 64)),
    ("bht,bthd->bhd", (2, 5, 1030), (2, 1030, 5, 72)),
    ("bht,bthd->dbh", (2, 5, 130), (2, 130, 5, 33)),
])
def test_matrix_vector_against_float64(eq, s0, s1, dtype):
    _check(eq, _rand(s0, dtype, 1), _rand(s1, dtype, 2))


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16])
@pytest.mark.parametrize("eq,s0,s1", [("ij,j->i", (130, 1024), (1024,)), ("i,ij->j", (600,), (600, 128))])
@pytest.mark.parametrize("off0,off1", [(1, 0), (0, 1), (3, 5)])
def test_bases_off_the_vector_grid(eq, s0, s1, off0, off1, dtype):
    _check(eq, _rand(s0, dtype, 3, off0), _rand(s1, dtype, 4, off1))


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16])
def test_special_values(dtype):
    """inf and NaN reach exactly the outputs whose sums hold them, subnormal
    operands are kept."""
    for eq, s0, s1 in (("ij,j->i", (300, 1030), (1030,)), ("i,ij->j", (1030,), (1030, 72))):
        a, b = _rand(s0, dtype, 5), _rand(s1, dtype, 6)
        m = a if a.dim() == 2 else b
        m[7, 3], m[20, 70], m[70, 5] = float("inf"), float("-inf"), float("nan")
        got, want = einsum(eq, a, b), torch.einsum(eq, a.double(), b.double())
        for f in (torch.isnan, torch.isposinf, torch.isneginf):
            assert torch.equal(f(got), f(want)), eq
        tiny = 2.0 ** -140 if dtype == torch.float32 else 2.0 ** -20
        a, b = (_rand(s0, dtype, 7).sign() * tiny).to(dtype), _rand(s1, dtype, 8)
        _check(eq, a, b)


def test_short_workspace_is_refused():
    K = 1 << 20
    d = launch.GemmDesc(dtype=launch.DT_F32, batch_shape=[], a_bstride=[], b_bstride=[], c_bstride=[], M=1, N=1, K=K,
                        a_ms=0, a_ks=1, b_ks=1, b_ns=0, c_ms=0, c_ns=0, a_numel=K, b_numel=K, c_numel=1)
    lib, cd = abi.bind(), abi.gemm_desc(d)
    need = int(lib.pe_gemm_workspace_bytes(ctypes.byref(cd)))
    x, out = torch.ones(K, device="cuda"), torch.zeros(1, device="cuda")
    assert need > 0
    ws = torch.empty(need, dtype=torch.uint8, device="cuda")
    args = [ctypes.c_void_p(t.data_ptr()) for t in (x, x, out, ws)]
    st = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    assert lib.pe_gemm(ctypes.byref(cd), *args, ctypes.c_int64(need - 1), st) == -4
    assert lib.pe_gemm(ctypes.byref(cd), *args, ctypes.c_int64(need), st) == 0
    assert float(out) == K


@pytest.mark.parametrize("eq,s0,s1", [("ij,j->i", (500, 32), (32,)), ("ij,j->i", (3, 29), (29,)),
                                      ("bi,bi->b", (300, 31), (300, 31)), ("bhd,bthd->bht", (2, 3, 9), (2, 70, 3, 9))])
def test_float16_short_rows_round_once(eq, s0, s1):
    """K <= 32: products and sums in 64 bits, one rounding to float32."""
    a, b = _rand(s0, torch.float16, 9), _rand(s1, torch.float16, 10)
    got, want = einsum(eq, a, b), torch.einsum(eq, a.double(), b.double())
    mag = torch.einsum(eq, a.double().abs(), b.double().abs())
    assert bool(((got.double() - want).abs() <= EPS * want.abs() + 2.0 ** -45 * mag).all())


@pytest.mark.parametrize("eq,s0,s1", [("bhd,bthd->bht", (4, 8, 64), (4, 500, 8, 64)),
                                      ("bhd,bthd->bht", (4, 8, 200), (4, 500, 8, 200)),
                                      ("i,ij->j", (512,), (512, 4096)), ("ij,j->i", (4096, 4096), (4096,))])
def test_float16_error_is_no_larger_than_the_tiles(eq, s0, s1):
    """Against 64 bits, next to the same sums as a product with two equal
    vectors (M or N of 2: matrix cores)."""
    a, b = _rand(s0, torch.float16, 11), _rand(s1, torch.float16, 12)
    want = torch.einsum(eq, a.double(), b.double())
    l, r = eq.split("->")[0].split(",")
    o = eq.split("->")[1]
    if len(l) <= len(r):
        two = einsum(l + "z," + r + "->" + o + "z", torch.stack([a, a], -1), b)
    else:
        two = einsum(l + "," + r + "z->" + o + "z", a, torch.stack([b, b], -1))
    e = [float((x.double() - want).norm() / want.norm()) for x in (einsum(eq, a, b), two[..., 0])]
    assert e[0] <= e[1], e


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16])
@pytest.mark.parametrize("eq,K,other", [("i,ij->j", k, 4096) for k in (8, 16, 24, 32, 48, 64, 256, 512, 1024)] +
                         [("ij,j->i", k, 4096) for k in (33, 48, 64)] +
                         [("bk,bkn->bn", k, 24) for k in (8, 9, 16, 33, 256)])
def test_error_is_no_larger_than_the_tiles(eq, K, other, dtype):
    """As test_float16_error_is_no_larger_than_the_tiles, where sums are short,
    split or met by many threads; over four inputs, and within the 1 % by which
    two such norms differ from sampling alone."""
    err = [0.0, 0.0]
    for seed in range(4):
        if eq == "ij,j->i":
            a, b = _rand((other, K), dtype, seed), _rand((K,), dtype, seed + 50)
            two = einsum("ij,jz->iz", a, torch.stack([b, b], -1))[..., 0]
        elif eq == "i,ij->j":
            a, b = _rand((K,), dtype, seed), _rand((K, other), dtype, seed + 50)
            two = einsum("iz,ij->jz", torch.stack([a, a], -1), b)[..., 0]
        else:
            a, b = _rand((500, K), dtype, seed), _rand((500, K, other), dtype, seed + 50)
            two = einsum("bkz,bkn->bnz", torch.stack([a, a], -1), b)[..., 0]
        want = torch.einsum(eq, a.double(), b.double())
        for i, x in enumerate((einsum(eq, a, b), two)):
            err[i] += float((x.double() - want).norm() / want.norm()) ** 2
    assert err[0] <= 1.01 ** 2 * err[1], [e ** 0.5 / 2 for e in err]
