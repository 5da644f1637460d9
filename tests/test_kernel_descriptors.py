"""Resources of the built gfx950 kernels, read from the library's kernel
descriptors."""
import re
import struct
import subprocess

import pytest

from pto_einsum import runtime

OBJDUMP = "/opt/rocm/llvm/bin/llvm-objdump"
MAGIC = b"__CLANG_OFFLOAD_BUNDLE__"


@pytest.fixture(scope="module")
def descriptors(tmp_path_factory):
    """{kernel: its descriptor's directives}"""
    data = open(runtime.core_library_path(), "rb").read()
    out, at = {}, data.find(MAGIC)
    while at >= 0:
        (n,) = struct.unpack_from("<Q", data, at + len(MAGIC))
        p = at + len(MAGIC) + 8
        for _ in range(n):
            off, size, idlen = struct.unpack_from("<QQQ", data, p)
            ident, p = data[p + 24:p + 24 + idlen], p + 24 + idlen
            if not ident.endswith(b"gfx950") or not size:
                continue
            co = tmp_path_factory.mktemp("co") / "kernels.co"
            co.write_bytes(data[at + off:at + off + size])
            text = subprocess.run([OBJDUMP, "-D", "-j", ".rodata", str(co)], check=True, capture_output=True,
                                  text=True).stdout
            out.update(re.findall(r"\.amdhsa_kernel (\S+)(.*?)\.end_amdhsa_kernel", text, re.S))
        at = data.find(MAGIC, p)
    return out


def test_no_kernel_reads_the_dispatch_packet(descriptors):
    """A per-lane array that the compiler puts into LDS is addressed with the
    block's size from the dispatch packet in host memory: a wave's first
    instruction then waits for that (10 us when all CUs ask)."""
    assert len(descriptors) > 300
    assert not [k for k, d in descriptors.items() if ".amdhsa_user_sgpr_dispatch_ptr 1" in d]
