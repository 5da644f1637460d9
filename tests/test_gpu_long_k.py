"""Contractions so long that a K range's end passes 2^31 in 32 bits: sums of
ones (exact in float32 through the vector kernels, whose partial sums are
multiples of 128) and the tile kernel for such K."""
import ctypes

import pytest
import torch

from pto_einsum import abi, launch, runtime

pytestmark = pytest.mark.gpu

K = 2 ** 31 - 128 * 800


@pytest.fixture(scope="module")
def ones():
    if torch.cuda.mem_get_info()[0] < 24 << 30:
        pytest.skip("needs 24 GiB of GPU memory")
    x = torch.ones(2 * K, dtype=torch.float16, device="cuda")
    yield x
    del x
    torch.cuda.empty_cache()


def _gemm(M, N, ones, **kw):
    d = abi.gemm_desc(launch.GemmDesc(
        dtype=launch.DT_F16, batch_shape=[], a_bstride=[], b_bstride=[], c_bstride=[], M=M, N=N, K=K, a_ms=K, a_ks=1,
        b_ks=1, b_ns=K, c_ms=N, c_ns=1, a_numel=M * K, b_numel=N * K, c_numel=M * N, **kw))
    lib, out = abi.bind(), torch.empty(M, N, device="cuda")
    ws = torch.empty(max(1, int(lib.pe_gemm_workspace_bytes(ctypes.byref(d)))), dtype=torch.uint8, device="cuda")
    # Both operands are the end of the same ones.
    a, b = (ones[(2 - n) * K:].data_ptr() for n in (M, N))
    rc = lib.pe_gemm(ctypes.byref(d), ctypes.c_void_p(a), ctypes.c_void_p(b), ctypes.c_void_p(out.data_ptr()),
                     ctypes.c_void_p(ws.data_ptr()), ctypes.c_int64(ws.numel()),
                     ctypes.c_void_p(torch.cuda.current_stream().cuda_stream))
    assert rc == 0, runtime.last_error()
    return out.double()


@pytest.mark.parametrize("M,N", [(1, 1), (1, 2)])
def test_dot_products(ones, M, N):
    assert torch.equal(_gemm(M, N, ones), torch.full((M, N), float(K), device="cuda", dtype=torch.float64))


def test_tiles(ones):
    """The 1024 partial sums (exact) are added in order: a rounding of at most
    64 each below 2^31."""
    got = _gemm(2, 2, ones, split_k=1024)
    assert bool(((got - K).abs() <= 1024 * 64).all()), got
