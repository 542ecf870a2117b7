"""Registers and scratch of the built FP32 kernels, from the metadata that the
compiler writes into their code objects: what decides how many waves a SIMD holds.
"""
import os
import struct

import msgpack
import pytest

from kmc_dn_amd import build

MAGIC = b"__CLANG_OFFLOAD_BUNDLE__"


def _code_objects(blob):
    """The gfx950 code objects of every offload bundle in the library."""
    at = blob.find(MAGIC)
    while at >= 0:
        n = struct.unpack_from("<Q", blob, at + len(MAGIC))[0]
        pos = at + len(MAGIC) + 8
        for _ in range(min(n, 16)):
            off, size, idlen = struct.unpack_from("<QQQ", blob, pos)
            name = blob[pos + 24:pos + 24 + idlen]
            pos += 24 + idlen
            if b"gfx950" in name and size:
                yield blob[at + off:at + off + size]
        at = blob.find(MAGIC, at + 1)


def _metadata(elf):
    """The AMDGPU metadata note (type 32) of a code object."""
    phoff = struct.unpack_from("<Q", elf, 32)[0]
    phsize, phnum = struct.unpack_from("<HH", elf, 54)
    for i in range(phnum):
        kind = struct.unpack_from("<I", elf, phoff + i * phsize)[0]
        off, size = struct.unpack_from("<Q16xQ", elf, phoff + i * phsize + 8)
        if kind != 4:   # PT_NOTE
            continue
        end = off + size
        while off + 12 <= end:
            namesz, descsz, kind = struct.unpack_from("<III", elf, off)
            desc = off + 12 + (namesz + 3) // 4 * 4
            if kind == 32:
                return msgpack.unpackb(elf[desc:desc + descsz], strict_map_key=False)
            off = desc + (descsz + 3) // 4 * 4
    return {}


@pytest.fixture(scope="module")
def kernels():
    if not os.path.exists(build.LIB):
        build.build()
    with open(build.LIB, "rb") as f:
        blob = f.read()
    out = {}
    for obj in _code_objects(blob):
        for k in _metadata(obj).get("amdhsa.kernels", []):
            out[k[".name"]] = k
    assert out, "no kernels found"
    return out


def _waves_per_simd(k):
    """512 registers per lane, granted in eights to VGPRs and AGPRs together."""
    used = -(-k[".vgpr_count"] // 8) * 8   # (the count holds the AGPRs)
    return 512 // used


def _named(kernels, stem):
    found = {n: k for n, k in kernels.items() if stem in n}
    assert found, stem
    return found


@pytest.mark.parametrize("chunks,waves", [(1, 4), (2, 4), (3, 3)])
def test_positions_kernels_hold_their_waves(kernels, chunks, waves):
    """Launches that fill the chip run these: 512 / VGPRs of them on a SIMD."""
    for name, k in _named(kernels, f"kmc_batch_pos_kernelILi{chunks}E").items():
        assert _waves_per_simd(k) >= waves, (name, k[".vgpr_count"])


@pytest.mark.parametrize("chunks", [1, 2, 3])
def test_table_kernels_keep_their_hop_loop_inline(kernels, chunks):
    """A hop loop called out of line reads its LDS tables by generic loads through
    pointers in scratch (hundreds of bytes a lane; spills alone are within 200)."""
    for name, k in _named(kernels, f"kmc_batch_fp32_kernelILi{chunks}E").items():
        assert k[".private_segment_fixed_size"] <= 200, name
        assert not k.get(".uses_dynamic_stack"), name
