"""Registers of the built kernels, read from the metadata of the library's own code objects: wavefronts per SIMD and registers in
scratch memory that the times of whole families of calls hang on, and that no comparison of results shows."""
import os
import re
import struct
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
MAGIC = b"__CLANG_OFFLOAD_BUNDLE__"


def _code_objects(data):
    at = data.find(MAGIC)
    while at >= 0:
        (n,) = struct.unpack_from("<Q", data, at + len(MAGIC))
        pos = at + len(MAGIC) + 8
        for _ in range(n):
            offset, size, length = struct.unpack_from("<QQQ", data, pos)
            if b"gfx950" in data[pos + 24:pos + 24 + length] and size:
                yield data[at + offset:at + offset + size]
            pos += 24 + length
        at = data.find(MAGIC, at + len(MAGIC))


def _metadata(elf):
    """The AMDGPU metadata note (name "AMDGPU", type 32) of a code object: a msgpack map."""
    import msgpack
    (shoff,) = struct.unpack_from("<Q", elf, 0x28)
    entsize, count = struct.unpack_from("<HH", elf, 0x3A)
    for k in range(count):
        kind, = struct.unpack_from("<I", elf, shoff + k * entsize + 4)
        if kind != 7:   # SHT_NOTE
            continue
        offset, size = struct.unpack_from("<QQ", elf, shoff + k * entsize + 0x18)
        pos, end = offset, offset + size
        while pos < end:
            namesz, descsz, ntype = struct.unpack_from("<III", elf, pos)
            desc = pos + 12 + (namesz + 3) // 4 * 4
            if elf[pos + 12:pos + 12 + 6] == b"AMDGPU" and ntype == 32:
                return msgpack.unpackb(elf[desc:desc + descsz], strict_map_key=False)
            pos = desc + (descsz + 3) // 4 * 4
    return {}


@pytest.fixture(scope="module")
def kernels():
    """{kernel as written in the sources: (VGPRs, VGPRs spilled)}"""
    from ncn_cuda_amd import _lib
    _lib.load()
    pytest.importorskip("msgpack")
    from ncn_cuda_amd._build import LIB_PATH
    with open(LIB_PATH, "rb") as fh:
        data = fh.read()
    found = [k for elf in _code_objects(data) for k in _metadata(elf).get("amdhsa.kernels", [])]
    names = subprocess.run(["c++filt"], input="\n".join(k[".name"] for k in found), capture_output=True, text=True).stdout.split("\n")
    return {n.replace("void ncn::", "").split("(")[0].replace(" ", ""): (k[".vgpr_count"], k[".vgpr_spill_count"]) for n, k in zip(names, found)}


def _at_most(kernels, pattern, vgprs, spilled, builds):
    mine = {n: v for n, v in kernels.items() if re.fullmatch(pattern, n)}
    assert len(mine) >= builds, (pattern, len(mine))
    worse = {n: v for n, v in mine.items() if v[0] > vgprs or v[1] > spilled}
    assert not worse, worse


def test_forward_on_wide_tiles_runs_three_waves(kernels):
    """Forward and inverse builds on tiles of 4 x 8, any type and activation, plain and gathered: 168 VGPRs are
    three waves per SIMD (one build for heads of one feature has always had two more)."""
    _at_most(kernels, r"stage_(forward|inverse)_kernel<\d+,\d+,4,8,\w+,\w+,-?\d>", 168, 0, 96)
    _at_most(kernels, r"headwise_forward_kernel<64,32,4,8,\w+,\w+,\w+>", 170, 0, 8)


def test_one_stage_backward_does_not_spill(kernels):
    """The backward builds on tiles of 4 x 4 with a wave for every tile, all types."""
    _at_most(kernels, r"stage_backward_kernel<\d+,\d+,4,4,true,false,false,(-1|0|1)>", 128, 0, 45)
    _at_most(kernels, r"stage_backward_kernel<\d+,\d+,4,4,true,true,false,(-1|0|1)>", 128, 1, 45)


def test_forward_windows_in_lds_run_two_workgroups(kernels):
    """Workgroups of 8 waves: 128 VGPRs are two to a CU."""
    _at_most(kernels, r"fused_forward_kernel<.*>", 128, 0, 96)


def test_other_activations_keep_their_waves(kernels):
    """Inverse builds for activations other than tanh on heads of one feature and tiles of 4 x 4, plain and gathered: five
    waves per SIMD (one build has always had one register more)."""
    _at_most(kernels, r"headwise_forward_kernel<\d+,\d+,4,4,false,true,\w+>", 97, 0, 20)
    _at_most(kernels, r"headwise_forward_kernel<\d+,\d+,4,4,false,true,true>", 96, 0, 10)


def test_backward_on_groups_of_two_heads_of_one_feature(kernels):
    """With a window for every workgroup (four registers have always spilled at heads laid out in eights), and looping over windows."""
    _at_most(kernels, r"pair_backward_kernel<\d+,true,\w+,false,true>", 128, 4, 6)
    _at_most(kernels, r"pair_backward_kernel<\d+,true,\w+,true,true>", 128, 18, 6)


def test_radix_backward_spills_little(kernels):
    _at_most(kernels, r"radix_backward_kernel<\d,\d+,true,false,false>", 128, 5, 10)


def test_odd_shapes_keep_their_waves(kernels):
    """Builds without priorities on tiles of 4 x 4 run five waves per SIMD, of 5 x 5 four."""
    _at_most(kernels, r"any_forward_kernel<4,4,\w+,\w+,\w+,false>", 96, 0, 8)
    _at_most(kernels, r"any_forward_kernel<5,5,\w+,\w+,\w+,false>", 128, 0, 8)
