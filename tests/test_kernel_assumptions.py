"""CPU check of what the compiled kernels are taken to be, from their descriptors in the built library (compiled here from
source): point and ray scattering address LDS from 0, so they have no static LDS, and form addresses as denormal floats,
which are not flushed."""
import struct
import subprocess

import pytest

from sfsim_amd import atmosphere as atm


def device_images():
    blob = open(atm.LIB_PATH, "rb").read()
    at = blob.find(b"__CLANG_OFFLOAD_BUNDLE__")
    while at >= 0:
        p = at + 32
        for _ in range(struct.unpack_from("<Q", blob, at + 24)[0]):
            offset, size, name = struct.unpack_from("<QQQ", blob, p)
            if b"gfx950" in blob[p + 24:p + 24 + name] and size:
                yield blob[at + offset:at + offset + size]
            p += 24 + name
        at = blob.find(b"__CLANG_OFFLOAD_BUNDLE__", at + 24)


def descriptors(elf):
    """{kernel: its 64-byte descriptor} of an AMDGPU code object."""
    shoff, = struct.unpack_from("<Q", elf, 40)
    shentsize, shnum = struct.unpack_from("<HH", elf, 58)
    sections = [struct.unpack_from("<IIQQQQIIQQ", elf, shoff + i * shentsize) for i in range(shnum)]
    found = {}
    for _, kind, _, _, offset, size, link, _, _, entsize in sections:
        if kind != 11:  # SHT_DYNSYM
            continue
        for i in range(size // entsize):
            name, _, _, shndx, value, _ = struct.unpack_from("<IBBHQQ", elf, offset + i * entsize)
            start = sections[link][4] + name
            symbol = elf[start:elf.index(b"\0", start)].decode()
            if symbol.endswith(".kd"):
                at = value - sections[shndx][3] + sections[shndx][4]
                found[symbol[:-3]] = elf[at:at + 64]
    return found


@pytest.fixture(scope="module")
def kernels():
    return {k: d for image in device_images() for k, d in descriptors(image).items()}


def test_lds_begins_at_zero_and_denormals_are_kept(kernels):
    names = [k for k in kernels if "point_scatter_kernel" in k or "18ray_scatter_kernel" in k]
    assert len(names) >= 44, subprocess.list2cmdline(sorted(kernels))
    for k in names:
        assert struct.unpack_from("<I", kernels[k], 0)[0] == 0, k  # group_segment_fixed_size
    for k, d in kernels.items():
        assert struct.unpack_from("<I", d, 48)[0] >> 16 & 3 == 3, k  # compute_pgm_rsrc1: FP32 denormals in and out
