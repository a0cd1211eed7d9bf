"""Scratch memory of the built kernels, from the metadata of the library's own code objects: a
kernel that spills inside its loop over keys loses what its layout won."""
import re
import struct
from pathlib import Path

import msgpack
import pytest

from omnia_amd import ops

LIB = Path(ops.__file__).with_name("_omnia_kernels.so")
MAGIC = b"__CLANG_OFFLOAD_BUNDLE__"


def _notes(elf: bytes):
    """AMDGPU metadata notes of a code object."""
    shoff, = struct.unpack_from("<Q", elf, 0x28)
    size, num = struct.unpack_from("<HH", elf, 0x3A)
    for i in range(num):
        _, kind, _, _, off, length = struct.unpack_from("<IIQQQQ", elf, shoff + i * size)
        at, end = off, off + length
        while kind == 7 and at < end:
            n, d, t = struct.unpack_from("<III", elf, at)
            at += 12 + (n + 3) // 4 * 4
            if t == 32:
                yield msgpack.unpackb(elf[at:at + d], strict_map_key=False)
            at += (d + 3) // 4 * 4


def scratch(pattern: str) -> dict:
    """Kernel name -> bytes of scratch a lane."""
    data, out = LIB.read_bytes(), {}
    for m in re.finditer(MAGIC, data):
        at = m.start() + len(MAGIC)
        num, = struct.unpack_from("<Q", data, at)
        at += 8
        for _ in range(num):
            off, size, length = struct.unpack_from("<QQQ", data, at)
            kind = data[at + 24:at + 24 + length]
            at += 24 + length
            if b"gfx950" in kind and size:
                for note in _notes(data[m.start() + off:m.start() + off + size]):
                    for k in note["amdhsa.kernels"]:
                        if re.search(pattern, k[".name"]):
                            out[k[".name"]] = k[".private_segment_fixed_size"]
    return out


@pytest.mark.skipif(not LIB.exists(), reason="the library is not built")
def test_prompt_attention_keeps_its_registers():
    """Heads of 128, windowed or not, kept keys or not, one group of waves or two: nothing in
    scratch (a capped kernel of two groups parks one register across its loop)."""
    got = scratch(r"prefill_kernelILi128ELi128ELb")
    assert len(got) == 10
    for name, size in got.items():
        assert size <= (8 if re.search(r"ELi1ELi2E", name) else 0), (name, size)
    assert not any(scratch("prefill_attn32_kernel").values())
