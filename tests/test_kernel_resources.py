"""Registers of the block kernels as the built library's code objects declare them: a kernel that
spills registers reloads them from memory inside its products, and the results do not show it.
The 256^3 forms of repeated products hold as many as their tiles need (208 and 112)."""
import os
import re
import struct

import pytest

import kami_amd

msgpack = pytest.importorskip("msgpack")

MAGIC = b"__CLANG_OFFLOAD_BUNDLE__"


def code_objects(data):
    at = data.find(MAGIC)
    while at >= 0:
        entry = at + 32
        for _ in range(struct.unpack_from("<Q", data, at + 24)[0]):
            off, size, length = struct.unpack_from("<QQQ", data, entry)
            if b"gfx950" in data[entry + 24:entry + 24 + length]:
                yield data[at + off:at + off + size]
            entry += 24 + length
        at = data.find(MAGIC, at + 24)


def kernels(elf):
    """Kernel descriptions in the note sections of an ELF64 code object."""
    sections, = struct.unpack_from("<Q", elf, 40)
    step, count = struct.unpack_from("<HH", elf, 58)
    for i in range(count):
        kind, = struct.unpack_from("<I", elf, sections + i * step + 4)
        at, size = struct.unpack_from("<QQ", elf, sections + i * step + 24)
        end = at + size
        while kind == 7 and at < end:
            name, desc, note = struct.unpack_from("<III", elf, at)
            at += 12 + (name + 3) // 4 * 4
            if note == 32:
                yield from msgpack.unpackb(elf[at:at + desc])["amdhsa.kernels"]
            at += (desc + 3) // 4 * 4


@pytest.fixture(scope="module")
def block_kernels():
    path = os.path.join(os.path.dirname(kami_amd.__file__), "libkami.so")
    data = open(path, "rb").read()
    found = {}
    for co in code_objects(data):
        for k in kernels(co):
            # block_gemm_kernel<Atom, BlockGeom<Atom, m, n, k, pm, pn, pk, ks, b>, ...>
            m = re.search(r"block_gemm_kernelI.*?BlockGeomI\w*?_((?:Li\d+E)+)E", k[".name"])
            if m:
                key = (tuple(int(x) for x in re.findall(r"Li(\d+)E", m[1])), "BF16" in k[".name"], k[".name"])
                found[key] = (k[".vgpr_count"], k[".vgpr_spill_count"])
    assert len(found) > 200
    return found


def test_repeated_256_holds_its_tiles_in_registers(block_kernels):
    for waves, most in ((8, 208), (16, 112)):
        forms = {k: v for k, v in block_kernels.items() if k[0][:7] == (256, 256, 256, waves, 1, 1, 256)}
        assert len(forms) == 4  # FP16 and BF16, B stored N x K and K x N
        for key, (registers, spilled) in forms.items():
            assert spilled == 0 and registers <= most, (key, registers, spilled)


def test_block_kernels_do_not_spill(block_kernels):
    # 16 waves on 256 x 256 x 32, and 224^3 K x N in its single stage: a few outside their products
    most = {(256, 256, 32, 16, 1, 1, 32): 10, (224, 224, 224, 14, 1, 1, 224): 2}
    for key, (_, spilled) in block_kernels.items():
        assert spilled <= most.get(key[0][:7], 0), (key, spilled)
