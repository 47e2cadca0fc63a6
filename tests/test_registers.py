"""Registers that the built kernels spill, read from the code objects in the
runtime library: a kernel that keeps spilling more pays for it in every tile."""
import os
import re
import struct
import sys

import msgpack
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, ROOT)
LIBRARY = os.path.join(ROOT, "onnx-mlir_amd", "csrc", "libom_mi355x.so")
MAGIC = b"__CLANG_OFFLOAD_BUNDLE__"


def _code_objects(blob):
    """The gfx950 ELF images of every offload bundle in the library."""
    at = blob.find(MAGIC)
    while at >= 0:
        count, = struct.unpack_from("<Q", blob, at + len(MAGIC))
        p = at + len(MAGIC) + 8
        for _ in range(count):
            offset, size, length = struct.unpack_from("<QQQ", blob, p)
            triple = blob[p + 24:p + 24 + length]
            p += 24 + length
            if b"gfx950" in triple and size:
                yield blob[at + offset:at + offset + size]
        at = blob.find(MAGIC, at + len(MAGIC))


def _kernels(elf):
    """The kernels' metadata (the AMDGPU note, a msgpack map)."""
    shoff, = struct.unpack_from("<Q", elf, 0x28)
    shentsize, shnum = struct.unpack_from("<HH", elf, 0x3A)
    for i in range(shnum):
        kind, = struct.unpack_from("<I", elf, shoff + i * shentsize + 4)
        if kind != 7:  # SHT_NOTE
            continue
        offset, size = struct.unpack_from("<QQ", elf, shoff + i * shentsize + 24)
        p, end = offset, offset + size
        while p + 12 <= end:
            nlen, dlen, ntype = struct.unpack_from("<III", elf, p)
            desc = p + 12 + (nlen + 3) // 4 * 4
            if ntype == 32:
                yield from msgpack.unpackb(elf[desc:desc + dlen], strict_map_key=False)["amdhsa.kernels"]
            p = desc + (dlen + 3) // 4 * 4


@pytest.fixture(scope="module")
def spills():
    """Mangled kernel name -> vector registers spilled."""
    if not os.path.exists(LIBRARY):
        import __graft_entry__
        __graft_entry__.build()
    blob = open(LIBRARY, "rb").read()
    found = {k[".name"]: k.get(".vgpr_spill_count", 0) for elf in _code_objects(blob) for k in _kernels(elf)}
    assert len(found) > 100
    return found


@pytest.mark.parametrize("kernel,most", [
    (r"k_gemm_i8_dmaI", 0),
    (r"k_gemm_i8_(dma_)?bsI", 0),  # every tile, with and without row sums, split
    (r"k_gemm_i8_wregI", 0),
    # any K, any alignment: two blocks of 128 x 128 a CU, or three of 64 x 128
    (r"k_gemm_i8ILi128ELi128ELi2ELi2ELi2E", 0),
    (r"k_gemm_i8ILi64ELi128ELi2ELi2ELi3E", 0),
    (r"k_gemm_i8_(skinny|batched|batched_flat|flight)I", 0),
    (r"k_(pad_rows|sum_parts|copy_in|copy_out|pack_b)", 0),
])
def test_kernels_spill_no_more_registers(spills, kernel, most):
    forms = {n: s for n, s in spills.items() if re.search(kernel, n)}
    for name in re.search(r"\((.*)\)I", kernel).group(1).split("|") if "(skinny" in kernel else ():
        assert any("k_gemm_i8_" + name + "I" in n for n in forms), name
    assert forms, sorted(spills)
    assert max(forms.values()) <= most, {n: s for n, s in forms.items() if s > most}
