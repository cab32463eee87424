"""What the compiler says of the kernels in the built libraries: registers, and scratch memory for those that did not fit."""
import os
import re
import struct
import subprocess

import msgpack
import pytest

from pulp_nn_amd import build

# kernels that hold more at once than one wave's registers would take if it were asked for all at the same place
FITTED = ("dwpw_kernel", "dwpw_chain_kernel", "dw_mfma_kernel")
MAGIC = b"__CLANG_OFFLOAD_BUNDLE__"


def _code_objects(lib):
    """The gfx950 code objects of a shared object that this repository's build linked: one bundle per translation unit."""
    data, at = open(lib, "rb").read(), 0
    while (at := data.find(MAGIC, at)) >= 0:
        count, pos = struct.unpack_from("<Q", data, at + len(MAGIC))[0], at + len(MAGIC) + 8
        for _ in range(count):
            off, size, n = struct.unpack_from("<QQQ", data, pos)
            name = data[pos + 24:pos + 24 + n]
            pos += 24 + n
            if b"gfx950" in name and size:
                yield data[at + off:at + off + size]
        at += len(MAGIC)


def _kernels(elf):
    """The kernels' entries in the metadata note of a code object."""
    shoff, shentsize, shnum = struct.unpack_from("<Q", elf, 0x28)[0], *struct.unpack_from("<HH", elf, 0x3A)
    for i in range(shnum):
        kind, off, size = struct.unpack_from("<I", elf, shoff + i * shentsize + 4)[0], *struct.unpack_from("<QQ", elf, shoff + i * shentsize + 0x18)
        end = off + size
        while kind == 7 and off + 12 <= end:
            namesz, descsz, what = struct.unpack_from("<III", elf, off)
            name = elf[off + 12:off + 12 + namesz]
            desc = off + 12 + (namesz + 3) // 4 * 4
            if what == 32 and name.startswith(b"AMDGPU"):
                yield from msgpack.unpackb(elf[desc:desc + descsz], strict_map_key=False)["amdhsa.kernels"]
            off = desc + (descsz + 3) // 4 * 4


def kernel_names(bn_bits):
    """Names of a library's kernels as a profiler prints them, without arguments."""
    names = [k[".name"] for elf in _code_objects(build.lib_path(bn_bits)) for k in _kernels(elf)]
    plain = subprocess.run(["c++filt"], input="\n".join(names), stdout=subprocess.PIPE, text=True, check=True).stdout.split("\n")
    return [n.removeprefix("void ").split("(")[0] for n in plain]


@pytest.mark.parametrize("bn_bits", [32, 64])
def test_no_vector_register_is_spilled(bn_bits):
    lib = build.lib_path(bn_bits)
    if not os.path.exists(lib):
        build.build(bn_bits)
    kernels = [k for elf in _code_objects(lib) for k in _kernels(elf)]
    for family in FITTED:
        assert any(family in k[".name"] for k in kernels), family
    spilled = {k[".name"]: k[".vgpr_spill_count"] for k in kernels if k[".vgpr_spill_count"] and any(f in k[".name"] for f in FITTED)}
    names = subprocess.run(["c++filt"], input="\n".join(spilled), stdout=subprocess.PIPE, text=True, check=True).stdout.split("\n")
    assert not spilled, "\n".join("%d registers: %s" % (n, s) for n, s in zip(spilled.values(), names))


@pytest.mark.parametrize("bn_bits", [32, 64])
def test_waves_of_small_depthwise_planes(bn_bits):
    """64 channels a workgroup: four workgroups share a compute unit with one or two MFMAs a unit, three with three."""
    kernels = {k[".name"]: k[".vgpr_count"] for elf in _code_objects(build.lib_path(bn_bits)) for k in _kernels(elf)}
    found = [(vgprs, {1: 128, 2: 128, 3: 168}.get(int(m[1]), 256), name) for name, vgprs in kernels.items()
             if (m := re.search(r"dw_mfma_kernelILi64ELi(\d+)E", name))]
    assert len(found) == 12 and not [f for f in found if f[0] > f[1]]


@pytest.mark.parametrize("bn_bits", [32, 64])
def test_waves_of_single_blocks(bn_bits):
    """Constants of 64 bits leave the kernels of a single block four waves a SIMD at least, those of one slice of weights five; so
    are the lean ones of the 32-bit library."""
    kernels = {k[".name"]: k[".vgpr_count"] for elf in _code_objects(build.lib_path(bn_bits)) for k in _kernels(elf)}
    blocks = [(m[1], m[2] == "1", vgprs) for name, vgprs in kernels.items()
              if (m := re.search(r"dwpw_kernelILi\d+ELi\d+ELi(\d+)ELb0ELb([01])E", name))]
    assert any(lean for _, lean, _ in blocks) == (bn_bits == 32)
    for slices, lean, vgprs in blocks:
        assert vgprs <= (96 if lean or (bn_bits == 64 and slices == "1") else 128), (slices, lean)
