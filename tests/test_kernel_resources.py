"""CPU check of the built library's kernel metadata (the code object notes the
compiler writes beside each kernel of csrc/): the varlen kernels keep the
workgroups per CU that their launch shapes assume."""
import re
import struct

import msgpack
import pytest

from voiceagent_amd.build import LIB_PATH

MAGIC = b"__CLANG_OFFLOAD_BUNDLE__"


def _code_objects(blob):
    at = blob.find(MAGIC)
    while at >= 0:
        (count,), pos = struct.unpack_from("<Q", blob, at + 24), at + 32
        for _ in range(count):
            off, size, name = struct.unpack_from("<QQQ", blob, pos)
            triple = blob[pos + 24:pos + 24 + name]
            pos += 24 + name
            if b"gfx950" in triple and size:
                yield blob[at + off:at + off + size]
        at = blob.find(MAGIC, pos)


def _metadata(elf):
    """amdhsa.kernels of one code object (ELF64, note type 32, msgpack)."""
    shoff, shsize, shnum = (struct.unpack_from("<Q", elf, 0x28)[0],
                            *struct.unpack_from("<HH", elf, 0x3A))
    for i in range(shnum):
        kind, = struct.unpack_from("<I", elf, shoff + i * shsize + 4)
        off, size = struct.unpack_from("<QQ", elf, shoff + i * shsize + 24)
        end = off + size
        while kind == 7 and off < end:  # SHT_NOTE
            name, desc, typ = struct.unpack_from("<III", elf, off)
            body = off + 12 + (name + 3) // 4 * 4
            if typ == 32:
                return msgpack.unpackb(elf[body:body + desc])["amdhsa.kernels"]
            off = body + (desc + 3) // 4 * 4
    return []


@pytest.fixture(scope="module")
def varlen_kernels():
    """{(bf16, D, G, causal, paged, once, f8, pro, split, half): VGPRs, LDS}"""
    found = {}
    for elf in _code_objects(LIB_PATH.read_bytes()):
        for k in _metadata(elf):
            m = re.match(r"_ZN2va23varlen_attention_kernelI(.*)EEvNS_12VarlenParamsE", k[".name"])
            if m:
                key = tuple(int(x) for x in re.findall(r"L[bi](\d+)E", m.group(1) + "E"))
                found[key] = (k[".vgpr_count"] + k.get(".agpr_count", 0),
                              k[".group_segment_fixed_size"])
    assert len(found) > 100
    return found


def test_varlen_workgroups_per_cu(varlen_kernels):
    # A SIMD has 512 registers of each lane, given out eight at a time, and a
    # workgroup is one wave on each SIMD; a CU has 160 KiB of LDS.  head_dim
    # 128 runs two workgroups, head_dim 64 three (four on 64-row items).
    short = {}
    for key, (vgprs, lds) in varlen_kernels.items():
        want = 2 if key[1] == 128 else (4 if key[9] else 3)
        have = min(512 // (-(-vgprs // 8) * 8), 160 * 1024 // lds)
        if have < want:
            short[key] = (vgprs, lds)
    assert not short
