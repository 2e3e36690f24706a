"""The registers of the counting kernels as compiled: what spills to scratch memory costs every call that
takes the kernel.  Read from the metadata of the built library's gfx950 code object, no GPU needed."""
import os
import struct

import msgpack
import pytest

import kcgpu_amd as K


def _code_objects(blob):
    """gfx950 ELF images of the offload bundles in a shared library"""
    magic, at = b"__CLANG_OFFLOAD_BUNDLE__", 0
    while (at := blob.find(magic, at)) >= 0:
        count, = struct.unpack_from("<Q", blob, at + len(magic))
        p = at + len(magic) + 8
        for _ in range(count):
            off, size, tlen = struct.unpack_from("<QQQ", blob, p)
            triple = blob[p + 24:p + 24 + tlen]
            p += 24 + tlen
            if b"gfx950" in triple and size:
                yield blob[at + off:at + off + size]
        at += len(magic)


def _kernels(elf):
    """{name: metadata} from the AMDGPU note of a code object"""
    shoff, = struct.unpack_from("<Q", elf, 40)
    shentsize, shnum = struct.unpack_from("<HH", elf, 58)
    for i in range(shnum):
        sh = shoff + i * shentsize
        if struct.unpack_from("<I", elf, sh + 4)[0] != 7:  # SHT_NOTE
            continue
        off, size = struct.unpack_from("<QQ", elf, sh + 24)
        namesz, descsz, _ = struct.unpack_from("<III", elf, off)
        desc = off + 12 + (namesz + 3) // 4 * 4
        meta = msgpack.unpackb(elf[desc:desc + descsz], strict_map_key=False)
        return {k[".name"]: k for k in meta["amdhsa.kernels"]}
    return {}


@pytest.fixture(scope="module")
def kernels():
    path = os.path.join(os.path.dirname(K.__file__), "libkcgpu.so")
    with open(path, "rb") as f:
        blob = f.read()
    out = {}
    for elf in _code_objects(blob):
        out.update(_kernels(elf))
    return out


def _named(kernels, part):
    found = {n: m for n, m in kernels.items() if part in n}
    assert found, part
    return found


def test_wide_kernel_keeps_its_registers(kernels):
    """the block-wide kernel (tasks above 256 vertices): no vector register spilled, few scalar ones; its instance for
    deep trees spills around the calls of its walks"""
    for name, m in _named(kernels, "k_pivot_wide").items():
        if "KindE4" not in name:
            assert m[".vgpr_spill_count"] == 0 and m[".sgpr_spill_count"] <= 200, name
            assert m[".private_segment_fixed_size"] <= 288, name
        else:
            assert m[".vgpr_spill_count"] <= 80 and m[".private_segment_fixed_size"] <= 640, name


def test_shallow_register_kernels_keep_their_registers(kernels):
    """the two- and four-word kernels without matrix operands: few registers spilled"""
    for part, spills in (("k_pivot_regILi2ELNS_4KindE1E", 60), ("k_pivot_regILi4ELNS_4KindE1E", 32)):
        for name, m in _named(kernels, part).items():
            assert m[".vgpr_spill_count"] <= spills, name


def test_resident_launch_keeps_its_registers(kernels):
    """the serving loop's resident kernel: eight waves per SIMD and no vector register spilled"""
    for name, m in _named(kernels, "k_pivot_open").items():
        assert m[".vgpr_count"] <= 64 and m[".vgpr_spill_count"] == 0, name
        assert m[".private_segment_fixed_size"] == 0, name


def test_generic_kernel_instances(kernels):
    """only the instances that a launch can take; the large classes' without the small ones' registers"""
    names = _named(kernels, "7k_countILb")
    assert len(names) == 8
    for part in ("7k_countILb0ELb0ELb0ELb0E", "7k_countILb0ELb1ELb0ELb0E"):
        for name, m in _named(kernels, part).items():
            assert m[".vgpr_count"] <= 64 and m[".private_segment_fixed_size"] == 0, name
