"""The compiled kernels of the built library, by their metadata and their assembly: what a
launch or a prologue must not pay for, though every result would still be right."""
import os
import re
import struct
import subprocess

import pytest

from jblas_amd import build as B

LLVM = os.path.join(os.path.dirname(os.path.dirname(B.HIPCC)), "llvm", "bin")
pytestmark = pytest.mark.skipif(not os.path.exists(os.path.join(LLVM, "llvm-objdump")) or not os.path.exists(B.LIB),
                                reason="needs the LLVM tools and the built library")


@pytest.fixture(scope="module")
def code_objects(tmp_path_factory):
    """The gfx950 code objects of the library, one per source file."""
    data, out, at = open(B.LIB, "rb").read(), [], 0
    while (at := data.find(b"__CLANG_OFFLOAD_BUNDLE__", at)) >= 0:
        pos = at + 32
        for _ in range(struct.unpack_from("<Q", data, at + 24)[0]):
            offset, size, n = struct.unpack_from("<QQQ", data, pos)
            name = data[pos + 24:pos + 24 + n].decode()
            pos += 24 + n
            if name.endswith(B.ARCH) and size:
                out.append(tmp_path_factory.mktemp("co") / f"{len(out)}.co")
                out[-1].write_bytes(data[at + offset:at + offset + size])
        at = pos
    assert out
    return out


def run(tool, *args):
    return subprocess.run([os.path.join(LLVM, tool), *map(str, args)], check=True, capture_output=True, text=True).stdout


def test_gemm_launches_without_implicit_arguments(code_objects):
    """A kernel that reads a grid or block dimension makes the host fill in 256 more bytes for every launch."""
    kernels = 0
    for co in code_objects:
        for k in run("llvm-readelf", "--notes", co).split(".agpr_count")[1:]:
            name = re.search(r"\.symbol:\s+(\S+)", k).group(1)
            if re.search("gemm_mfma_kernel|fastmul|grouped_ring_kernel|grouped_x3_kernel", name):
                kernels += 1
                assert "hidden_" not in k, name
    assert kernels >= 40


def test_ring_loads_have_scalar_descriptors(code_objects):
    """A buffer descriptor in vector registers is loaded through in a loop over its values (exec is narrowed to the
    lanes of one value and the rest go round again)."""
    kernels = 0
    for co in code_objects:
        if "ring_kernel" not in (symbols := run("llvm-readelf", "--symbols", "--wide", co)) and "gemm_mfma_kernel" not in symbols:
            continue
        for f in run("llvm-objdump", "-d", "--no-show-raw-insn", co).split("\n\n"):
            if re.search("gemm_mfma_kernel|grouped_ring_kernel", f.split("\n", 1)[0]):
                kernels += 1
                assert not re.search(r"s_xor_b64 exec, exec", f), f.split("\n", 1)[0]
    assert kernels >= 40
