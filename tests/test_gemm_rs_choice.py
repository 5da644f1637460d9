"""Which GEMMs take the register-staged kernel, read on the CPU through
pe_gemm_choice (float32: a rule on extents and strides alone), and the loads of
that kernel emulated: every vector inside its operand."""
import ctypes

import pytest

from pto_einsum import abi, launch


def _choice(M, N, K, nb=1, al="k", bl="n", dtype=launch.DT_F32):
    d = launch.GemmDesc(dtype=dtype, batch_shape=[nb], a_bstride=[M * K], b_bstride=[K * N], c_bstride=[M * N],
                        M=M, N=N, K=K, a_ms=K if al == "k" else 1, a_ks=1 if al == "k" else M,
                        b_ks=N if bl == "n" else 1, b_ns=1 if bl == "n" else K, c_ms=N, c_ns=1,
                        a_numel=nb * M * K, b_numel=nb * K * N, c_numel=nb * M * N)
    lib, cd, info = abi.bind(), abi.gemm_desc(d), (ctypes.c_int64 * 4)()
    assert lib.pe_gemm_choice(ctypes.byref(cd), info) == 0
    return list(info), int(lib.pe_gemm_workspace_bytes(ctypes.byref(cd)))


@pytest.mark.parametrize("shape,nb,want", [
    ((2048, 2048, 512), 1, [128, 128, 1, 512]),     # 256 tiles: one per CU (64x64 float32 tiles before)
    ((256, 256, 256), 64, [128, 128, 1, 256]),
    ((1664, 1920, 1000), 1, [128, 128, 1, 1000]),   # 195 tiles unsplit rather than 3 splits of them
    ((4096, 128, 4096), 1, [128, 128, 16, 256]),
    ((384, 2816, 1536), 1, [64, 64, 6, 256]),       # 66 tiles: the float32 kernel keeps it
    ((128, 128, 128), 1024, [128, 128, 1, 128]),    # short K: the float32 kernel's tile
])
def test_float32_choice_and_workspace(shape, nb, want):
    info, ws = _choice(*shape, nb=nb)
    assert info == want
    assert ws == (info[2] * nb * shape[0] * shape[1] * 4 if info[2] > 1 else 0)


def _addresses(L, V, rows_tile, BK, rows, K, kps):
    """(address, length) of every vector load of the kernel for one operand of
    `rows` x K, contiguous along k (L = "k") or rows, as pe_gemm_rs.h forms
    them."""
    vpr = BK // V if L == "k" else rows_tile // V
    step, nv = 256 // vpr, rows_tile * BK // V // 256
    rs, ks = (K, 1) if L == "k" else (1, rows)
    for tm in range(-(-rows // rows_tile)):
        left = rows - tm * rows_tile
        back = rows_tile - left if L == "n" and left < rows_tile and left % V and tm > 0 else 0
        m0 = tm * rows_tile - back
        left = rows - m0
        whole = L == "k" or left >= rows_tile or left % V == 0
        for kb in range(0, K, kps):
            klen = min(K, kb + kps) - kb
            ns = -(-klen // BK)
            first = klen - (ns - 1) * BK
            for s in range(ns):
                k0, kn = (0, first) if s == 0 else (first + (s - 1) * BK, BK)
                base = m0 * rs + (kb + k0) * ks
                for tid in range(256):
                    for v in range(nv):
                        p, c = tid // vpr + v * step, (tid % vpr) * V
                        r, k = (p, c) if L == "k" else (c, p)
                        if s == 0 or not whole:
                            if L == "k":
                                yield base + min(r, left - 1) * rs + max(min(k, kn - V), -(kb + k0)), V
                            else:
                                yield base + min(k, kn - 1) * ks + min(r, left - V), V
                        else:
                            r = min(r, left - 1) if L == "k" else max(0, min(r, left - V))
                            yield base + r * rs + k * ks, V


@pytest.mark.parametrize("V,rows_tile,BK", [(4, 128, 16), (8, 128, 64), (8, 64, 32)])
@pytest.mark.parametrize("rows,K", [(8, 8), (63, 9), (129, 65), (131, 63), (136, 129), (200, 17), (257, 81)])
@pytest.mark.parametrize("L", ["k", "n"])
def test_every_load_lies_in_its_operand(L, V, rows_tile, BK, rows, K):
    for kps in (K, 64):
        for addr, n in _addresses(L, V, rows_tile, BK, rows, K, kps):
            assert 0 <= addr and addr + n <= rows * K


@pytest.mark.parametrize("dtype", [launch.DT_F16, launch.DT_F32])
@pytest.mark.parametrize("M,N,K", [(640, 48, 1992), (768, 96, 560), (304, 200, 1000), (504, 536, 504), (4000, 128, 4104),
                                   (264, 264, 1960), (2000, 3000, 72), (1000, 1504, 160), (2048, 2048, 512),
                                   (1664, 1920, 1000), (136, 264, 200)])
def test_split_does_not_depend_on_alignment(M, N, K, dtype):
    """Operands off the vector grid (as an odd batch stride of one batch makes
    them for the choice) are split as aligned ones are, where those are split
    or unsplit by the same rule."""
    infos = []
    for odd in (0, 1):
        d = launch.GemmDesc(dtype=dtype, batch_shape=[1], a_bstride=[M * K + odd], b_bstride=[K * N + odd],
                            c_bstride=[M * N], M=M, N=N, K=K, a_ms=K, a_ks=1, b_ks=N, b_ns=1, c_ms=N, c_ns=1,
                            a_numel=M * K, b_numel=K * N, c_numel=M * N)
        lib, cd, info = abi.bind(), abi.gemm_desc(d), (ctypes.c_int64 * 4)()
        assert lib.pe_gemm_choice(ctypes.byref(cd), info) == 0
        infos.append(([info[2], info[3] if info[2] > 1 else K], int(lib.pe_gemm_workspace_bytes(ctypes.byref(cd)))))
        assert infos[-1][1] >= (infos[-1][0][0] * M * N * 4 if infos[-1][0][0] > 1 else 0)
    assert infos[0] == infos[1]


@pytest.mark.parametrize("nb,M,N,K,al,bl,taken", [
    (100, 130, 260, 256, "k", "n", False), (82, 152, 400, 512, "n", "n", False), (37, 132, 1000, 1024, "k", "k", False),
    (4, 1040, 1040, 256, "n", "n", False), (60, 384, 384, 256, "n", "n", True), (16, 1000, 1536, 777, "n", "n", True),
    (100, 130, 260, 257, "k", "n", False), (3, 1025, 1023, 101, "k", "n", True), (90, 129, 255, 65, "n", "k", False),
])
def test_float32_padding_rule(nb, M, N, K, al, bl, taken):
    """Its 128x128 tiles only where they cover little more than 64x64 ones: 1.1
    times, 1.3 for extents that the direct-load kernel cannot take."""
    info, ws = _choice(M, N, K, nb=nb, al=al, bl=bl)
    assert info[2] == 1 and ws == 0
    assert (info[:2] == [128, 128]) == taken
