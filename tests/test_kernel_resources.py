"""The library's kernels keep their values in registers: no private segment (scratch memory in HBM), read from the
metadata that the compiler writes into the library's own code objects.  The exceptions are the split-context kernels on
token pages at F32 head_dim 128, which spill 6 registers beside their loop.

Beside the time it costs, a spill has given wrong results here: a merge kernel with 8 partial rows in flight at F32
head_dim 224 spilled a 16-byte value as 12 bytes in scratch and 4 in an accumulation register, and the reload left
the last 4 out."""
import os
import struct

import pytest

msgpack = pytest.importorskip("msgpack")

LIB = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "mini-vllm-rs_amd", "libmvr_attn.so")
MAGIC = b"__CLANG_OFFLOAD_BUNDLE__"
NT_AMDGPU_METADATA = 32


def code_objects(data):
    """The gfx950 ELF images of every offload bundle in the library."""
    at = data.find(MAGIC)
    while at >= 0:
        (count,) = struct.unpack_from("<Q", data, at + len(MAGIC))
        pos = at + len(MAGIC) + 8
        for _ in range(count):
            offset, size, name = struct.unpack_from("<QQQ", data, pos)
            target = data[pos + 24:pos + 24 + name]
            pos += 24 + name
            if b"gfx950" in target and size:
                yield data[at + offset:at + offset + size]
        at = data.find(MAGIC, at + 1)


def kernels(elf):
    (shoff,) = struct.unpack_from("<Q", elf, 40)
    entry, num = struct.unpack_from("<HH", elf, 58)
    for i in range(num):
        kind, _, _, offset, size = struct.unpack_from("<IQQQQ", elf, shoff + i * entry + 4)
        while kind == 7 and size > 0:  # SHT_NOTE
            n, d, note = struct.unpack_from("<III", elf, offset)
            name, desc = offset + 12, offset + 12 + -(-n // 4) * 4
            if note == NT_AMDGPU_METADATA and elf[name:name + 6] == b"AMDGPU":
                yield from msgpack.unpackb(elf[desc:desc + d], strict_map_key=False)["amdhsa.kernels"]
            step = 12 + -(-n // 4) * 4 + -(-d // 4) * 4
            offset, size = offset + step, size - step


def test_no_kernel_spills_to_scratch():
    if not os.path.exists(LIB):
        pytest.skip("build the library first (python -c 'import __graft_entry__ as g; g.build()')")
    found = [k for elf in code_objects(open(LIB, "rb").read()) for k in kernels(elf)]
    names = {k[".name"] for k in found}
    assert len(names) > 100 and any("paged_prefill" in n for n in names) and any("merge" in n for n in names)
    spilled = {k[".name"]: k[".vgpr_spill_count"] for k in found
               if k[".private_segment_fixed_size"] or k[".vgpr_spill_count"]}
    token_pages = {n for n in spilled if "paged_attention_kernelINS0_9F32TraitsILi128E" in n and "ELi1ELb1EEEv" in n}
    assert set(spilled) <= token_pages, spilled
    assert all(n <= 6 for n in spilled.values()), spilled
