"""Which GEMMs take the register-staged kernel, read on the CPU through
pe_gemm_choice (float32: a rule on extents and strides alone), and that
kernel's loads, run on the CPU: every vector inside its operand."""
import ctypes
import os
import subprocess

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


@pytest.fixture(scope="module")
def loads(tmp_path_factory):
    """rs_loads.hip: the kernel's own load functions, built for the CPU."""
    here = os.path.dirname(os.path.abspath(__file__))
    exe = tmp_path_factory.mktemp("loads") / "rs_loads"
    subprocess.run(["/opt/rocm/bin/hipcc", "-x", "hip", "--offload-host-only", "-O1", "-std=c++17", "-w",
                    "-I" + os.path.join(here, "..", "include"),
                    "-I" + os.path.join(here, "..", "pto-einsum_amd", "csrc"), os.path.join(here, "rs_loads.hip"),
                    "-o", str(exe)], check=True)
    return str(exe)


@pytest.mark.parametrize("V,rows_tile,BK", [(4, 128, 16), (8, 128, 64), (8, 64, 32)])
@pytest.mark.parametrize("rows,K", [(8, 8), (63, 9), (129, 65), (131, 63), (136, 129), (200, 17), (257, 81)])
@pytest.mark.parametrize("L", ["k", "n"])
def test_every_load_lies_in_its_operand(loads, L, V, rows_tile, BK, rows, K):
    """... between inaccessible pages, and delivers its elements, zeros past K."""
    r = subprocess.run([loads, str(V), str(rows_tile), L, str(rows), str(K)], capture_output=True, text=True)
    assert r.returncode == 0, (r.returncode, r.stdout)


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
