"""Registers and scratch memory of the built kernels, read from the code objects
in the library.  The kernels for mechanisms whose reactions are all standard
hold nothing of the general code: no registers saved around calls that they
never make, and wavefronts per SIMD as their launch bounds ask for."""
import re
import struct

import msgpack
import pytest

MAGIC = b"__CLANG_OFFLOAD_BUNDLE__"


def notes(elf):
    """(type, description) of the notes of a 64-bit little-endian ELF file."""
    phoff, = struct.unpack_from("<Q", elf, 32)
    phentsize, phnum = struct.unpack_from("<HH", elf, 54)
    for i in range(phnum):
        ptype, _, off, _, _, size = struct.unpack_from("<IIQQQQ", elf, phoff + i * phentsize)
        p, end = off, off + size
        while ptype == 4 and p + 12 <= end:
            nlen, dlen, kind = struct.unpack_from("<III", elf, p)
            d = p + 12 + (nlen + 3) // 4 * 4
            yield kind, elf[d:d + dlen]
            p = d + (dlen + 3) // 4 * 4


@pytest.fixture(scope="module")
def kernels():
    from cantera_amd._lib import LIB_PATH
    lib = open(LIB_PATH, "rb").read()
    found = {}
    for m in re.finditer(re.escape(MAGIC), lib):
        base = m.start()
        p = base + len(MAGIC) + 8
        for _ in range(struct.unpack_from("<Q", lib, p - 8)[0]):
            off, size, tlen = struct.unpack_from("<QQQ", lib, p)
            triple = lib[p + 24:p + 24 + tlen]
            p += 24 + tlen
            if b"gfx950" not in triple or not size:
                continue
            for kind, desc in notes(lib[base + off:base + off + size]):
                if kind == 32:   # NT_AMDGPU_METADATA
                    for k in msgpack.unpackb(desc)["amdhsa.kernels"]:
                        found[k[".name"]] = k
    assert found
    return found


def pick(kernels, pattern):
    k = [v for name, v in kernels.items() if re.search(pattern, name)]
    assert k, pattern
    return k


@pytest.mark.parametrize("pattern,scratch,vgprs", [
    # one state per wavefront, FP64 constants: three wavefronts per SIMD
    (r"\d+rates_kernelILi[12]ELb0ELb0E", 0, 168),
    (r"reactor_rates_kernelILi[12]ELb0E", 0, 168),
    # Jacobians: two wavefronts per SIMD (512 registers of a lane)
    (r"jac_batch_kernelI", 64, 256),
    # integrators of h2o2, gri30 and n-dodecane (their own frames)
    (r"bdf_advance_r16IdLb0ELb0E", 240, 512),
    (r"bdf_advance_lr56IdLb0ELb0E", 280, 512),
    (r"bdf_advance_moleILi2ELb0E", 290, 512),
])
def test_no_general_code(kernels, pattern, scratch, vgprs):
    for k in pick(kernels, pattern):
        assert k[".private_segment_fixed_size"] <= scratch, k[".name"]
        assert k[".vgpr_count"] <= vgprs, k[".name"]


def test_equilibrium_two_wavefronts_per_simd(kernels):
    """Eight wavefronts of a CU in its 160 KB of LDS and 512 registers a lane."""
    for k in pick(kernels, r"equil_kernelILi[12]E"):
        assert k[".vgpr_count"] <= 256, k[".name"]
        assert k[".group_segment_fixed_size"] <= 160 * 1024 // 8, k[".name"]
