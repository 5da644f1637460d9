"""K ranges and slab counts of the kernels (pe_ranges.h, the header that they
include, built here for the CPU) at extents up to the largest that descriptors
accept, with the splits that the library chooses for them."""
import ctypes
import os
import subprocess

import pytest

from pto_einsum import abi, launch

CSRC = os.path.join(os.path.dirname(os.path.abspath(__file__)), "..", "pto-einsum_amd", "csrc")
TOP = 2 ** 31 - 1


@pytest.fixture(scope="module")
def ranges(tmp_path_factory):
    d = tmp_path_factory.mktemp("ranges")
    src, lib = d / "ranges.cpp", d / "libranges.so"
    src.write_text('#include "pe_ranges.h"\nextern "C" {\n'
                   "int k_range(int K, int kb, int per) { return pe::k_range(K, kb, per); }\n"
                   "int k_slabs(int len, int bk) { return pe::k_slabs(len, bk); }\n"
                   "bool k_ends_fit(int64_t K) { return pe::k_ends_fit(K); }\n"
                   "int64_t product_tile_blocks(int64_t P, int64_t Q, int64_t b)"
                   " { return pe::product_tile_blocks(P, Q, b); }\n"
                   "int64_t axis_part(int64_t n) { return pe::axis_part(n); }\n"
                   "unsigned next_index(unsigned i, unsigned s, unsigned n) { return pe::next_index(i, s, n); }\n}\n")
    # -fwrapv: 32-bit sums wrap, as they do on the GPU.
    subprocess.run(["g++", "-std=c++17", "-O1", "-fwrapv", "-shared", "-fPIC", f"-I{CSRC}", str(src), "-o", str(lib)],
                   check=True)
    lib = ctypes.CDLL(str(lib))
    lib.next_index.restype, lib.axis_part.restype = ctypes.c_uint32, ctypes.c_int64
    lib.k_ends_fit.restype = ctypes.c_bool
    lib.product_tile_blocks.restype = ctypes.c_int64
    lib.product_tile_blocks.argtypes = [ctypes.c_int64] * 3
    return lib


def _choice(M, N, K, dtype, bl="k", split_k=0, tile=0):
    d = launch.GemmDesc(dtype=dtype, batch_shape=[], a_bstride=[], b_bstride=[], c_bstride=[], M=M, N=N, K=K,
                        a_ms=K, a_ks=1, b_ks=1 if bl == "k" else N, b_ns=K if bl == "k" else 1, c_ms=N, c_ns=1,
                        a_numel=M * K, b_numel=K * N, c_numel=M * N, split_k=split_k, tile=tile)
    info = (ctypes.c_int64 * 4)()
    assert abi.bind().pe_gemm_choice(ctypes.byref(abi.gemm_desc(d)), info) == 0
    return list(info)


@pytest.mark.parametrize("dtype", [launch.DT_F32, launch.DT_F16])
@pytest.mark.parametrize("K", [TOP, TOP - 7, 2 ** 31 - 64, 2 ** 31 - 100000, 2 ** 31 - 262145, 2 ** 31 - 524289,
                               2 ** 31 - 2 ** 20 - 8,
                               2 ** 30 + 1, 1000003, 4096, 77])
@pytest.mark.parametrize("M,N,bl,split_k,tile", [
    (1, 1, "k", 0, 0),       # a dot product: up to 1024 ranges
    (1, 8, "n", 0, 0),       # vector times matrix
    (2, 3, "k", 0, 0),       # matrix cores
    (2, 3, "k", 1, 0), (2, 3, "k", 7, 64), (200, 200, "n", 1, 128),
])
def test_k_ranges_tile_the_contraction(ranges, M, N, bl, split_k, tile, K, dtype):
    _, _, split, per = _choice(M, N, K, dtype, bl, split_k, tile)
    assert 1 <= split and 0 < per <= TOP
    at = 0
    for s in range(split):
        assert s * per == at <= TOP                  # the kernels' 32-bit start
        n = ranges.k_range(K, s * per, per)
        assert 0 < n <= per
        for bk in (16, 32, 64):
            assert ranges.k_slabs(n, bk) == -(-n // bk)
        at += n
    assert at == K
    if ranges.k_ends_fit(ctypes.c_int64(K)):
        assert split * per <= TOP and K + 255 <= TOP


@pytest.mark.parametrize("n", [TOP, TOP - 7, 2 ** 31 - 128, 2 ** 31 - 255, 2 ** 31 - 256, 2 ** 31 - 257, 2 ** 30, 1])
def test_tiles_of_a_launch_end_below_the_32_bit_range(ranges, n):
    first = ranges.axis_part(ctypes.c_int64(n))
    assert 0 < first <= n
    for part in {first, n - first}:
        for tile in (32, 64, 128, 192, 256):
            assert -(-part // tile) * tile <= TOP


@pytest.mark.parametrize("n", [2 ** 32 - 1, 2 ** 32 - 2 ** 19, 2 ** 32 - 2 ** 19 - 1, 2 ** 19, 2 ** 19 + 1, 5])
def test_strided_walks_end(ranges, n):
    stride = 2048 * 256
    for first in (0, 3, min(n, stride) - 1):
        last = first + (n - 1 - first) // stride * stride if first < n else first
        if first < n:
            assert ranges.next_index(ctypes.c_uint32(last), ctypes.c_uint32(stride), ctypes.c_uint32(n)) == n
        if last > first:
            assert ranges.next_index(ctypes.c_uint32(first), ctypes.c_uint32(stride), ctypes.c_uint32(n)) == first + stride


@pytest.mark.parametrize("P,Q,batches,want", [
    (4096, 4096, 1, 4096), (1001, 1003, 3, 768), (16, 16, 1000, 1000), (8, 64, 7, 7), (8, 1024, 7, 112),
    (65, 65, 2, 8), (8, 65, 1, 2),
    (64, 64, (1 << 24) - 1, (1 << 24) - 1), (64, 64, 1 << 24, 0), (8, 65, 1 << 23, 0),    # 2^32 threads
    (8, 8, 1 << 20, 0), (12, 12, 1000, 0), (15, 17, 3, 0), (9, 513, 1, 9), (8, 31, 5, 0),     # mostly empty tiles
])
def test_product_tiles_are_filled_and_fit_a_launch(ranges, P, Q, batches, want):
    assert ranges.product_tile_blocks(P, Q, batches) == want


@pytest.mark.parametrize("dtype", [launch.DT_F32, launch.DT_F16])
@pytest.mark.parametrize("nb,N,K,bl,taken", [
    (2 ** 24 - 1, 8, 8, "n", True), (2 ** 24, 8, 8, "n", False),    # a block for each batch
    (2 ** 24, 16, 300, "k", False), (2 ** 22 - 1, 16, 300, "k", True),    # four rows of a batch in a block
    (2 ** 24, 2, 200, "k", True),                                         # 64 rows of any batch
])
def test_vector_kernels_fit_a_launch(nb, N, K, bl, taken, dtype):
    """Grids of 2^32 threads stay on the tile kernels, which walk a smaller one."""
    if bl == "k" and dtype == launch.DT_F32:
        K //= 2     # the same lanes for each row
    d = launch.GemmDesc(dtype=dtype, batch_shape=[nb], a_bstride=[K], b_bstride=[K * N], c_bstride=[N], M=1, N=N, K=K,
                        a_ms=0, a_ks=1, b_ks=1 if bl == "k" else N, b_ns=K if bl == "k" else 1, c_ms=0, c_ns=1,
                        a_numel=nb * K, b_numel=nb * K * N, c_numel=nb * N)
    info = (ctypes.c_int64 * 4)()
    assert abi.bind().pe_gemm_choice(ctypes.byref(abi.gemm_desc(d)), info) == 0
    assert (list(info)[:2] == [1, 1]) == taken
