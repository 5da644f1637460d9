"""GEMMs whose output is contiguous along M: the operands exchange their roles
(pe_gemm), at odd sizes, in every operand layout, with batches and K splits,
against float64; and the CPU's view of the same descriptors."""
import ctypes

import pytest
import torch

from pto_einsum import abi, launch

EPS = 2.0 ** -24


def _desc(nb, M, N, K, al, bl, dtype, out_m, **kw):
    return launch.GemmDesc(dtype=dtype, batch_shape=[nb], a_bstride=[M * K], b_bstride=[K * N], c_bstride=[M * N],
                           M=M, N=N, K=K, a_ms=K if al == "k" else 1, a_ks=1 if al == "k" else M,
                           b_ks=N if bl == "n" else 1, b_ns=1 if bl == "n" else K,
                           c_ms=1 if out_m else N, c_ns=M if out_m else 1,
                           a_numel=nb * M * K, b_numel=nb * K * N, c_numel=nb * M * N, **kw)


def _info(d):
    lib, cd, info = abi.bind(), abi.gemm_desc(d), (ctypes.c_int64 * 4)()
    assert lib.pe_gemm_choice(ctypes.byref(cd), info) == 0
    return list(info), int(lib.pe_gemm_workspace_bytes(ctypes.byref(cd)))


SIZES = [(3, 65, 33, 40), (2, 130, 257, 64), (1, 256, 1024, 512), (40, 129, 131, 193), (1, 96, 80, 5000), (1, 7, 9, 3),
         (1, 512, 512, 4096), (2, 1, 300, 64), (2, 300, 1, 64), (1, 2048, 1280, 128)]


@pytest.mark.parametrize("dtype", [launch.DT_F32, launch.DT_F16])
@pytest.mark.parametrize("al", ["k", "m"])
@pytest.mark.parametrize("bl", ["n", "k"])
@pytest.mark.parametrize("nb,M,N,K", SIZES)
def test_choice_is_the_exchanged_product_s(nb, M, N, K, al, bl, dtype):
    """Tile, split and workspace are those of C' = B' A'."""
    info, ws = _info(_desc(nb, M, N, K, al, bl, dtype, True))
    x = _desc(nb, N, M, K, "k" if bl == "k" else "m", "n" if al == "m" else "k", dtype, False)
    if M != 1 and N != 1:
        want, wx = _info(x)
        assert [info[1], info[0]] + info[2:] == want and ws == wx
    # An explicit tile keeps the roles that the caller gave.
    fixed, _ = _info(_desc(nb, M, N, K, al, bl, dtype, True, tile=64, split_k=2))
    assert fixed[:2] == [64, 64]


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [launch.DT_F32, launch.DT_F16])
@pytest.mark.parametrize("al", ["k", "m"])
@pytest.mark.parametrize("bl", ["n", "k"])
@pytest.mark.parametrize("nb,M,N,K", SIZES)
def test_output_along_m(nb, M, N, K, al, bl, dtype):
    """K roundings of sum |a||b| each, with exactly the workspace asked for;
    a guard after the output stays."""
    g = torch.Generator().manual_seed(M + N + K)
    dt = torch.float32 if dtype == launch.DT_F32 else torch.float16
    a = torch.randn((nb, M, K) if al == "k" else (nb, K, M), generator=g).to(dt).cuda()
    b = torch.randn((nb, K, N) if bl == "n" else (nb, N, K), generator=g).to(dt).cuda()
    d = abi.gemm_desc(_desc(nb, M, N, K, al, bl, dtype, True))
    lib = abi.bind()
    need = int(lib.pe_gemm_workspace_bytes(ctypes.byref(d)))
    ws = torch.empty(max(need, 16), dtype=torch.uint8, device="cuda")
    out = torch.full((nb * M * N + 64,), 7.0, device="cuda")
    args = [ctypes.c_void_p(t.data_ptr()) for t in (a, b, out, ws)]
    st = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    assert lib.pe_gemm(ctypes.byref(d), *args, ctypes.c_int64(need), st) == 0
    A = (a if al == "k" else a.transpose(1, 2)).double().contiguous()
    B = (b if bl == "n" else b.transpose(1, 2)).double().contiguous()
    got = out[:nb * M * N].view(nb, N, M).transpose(1, 2).double()
    assert bool(((got - torch.bmm(A, B)).abs() <= K * EPS * torch.bmm(A.abs(), B.abs())).all())
    assert bool((out[nb * M * N:] == 7.0).all())
