"""Registers and scratch memory of the persistent kernels, from the built library's kernel metadata.

A SIMD's 512 vector registers are shared by its waves, and a kernel's registers are those of its
largest path: one path that keeps too many units in flight costs every plan its occupancy.
"""

import os
import struct

import pytest

from elasticmegatron_amd import build

MAGIC = b"__CLANG_OFFLOAD_BUNDLE__"
SHT_NOTE = 7


def _kernels(path):
    """Metadata of every gfx950 kernel of a library: name -> its entry of the code object's note."""
    msgpack = pytest.importorskip("msgpack")
    with open(path, "rb") as f:
        d = f.read()
    out, pos = {}, d.find(MAGIC)
    while pos >= 0:
        n, = struct.unpack_from("<Q", d, pos + 24)
        p = pos + 32
        for _ in range(n):
            off, size, ln = struct.unpack_from("<QQQ", d, p)
            target = d[p + 24:p + 24 + ln]
            p += 24 + ln
            if b"gfx950" not in target or not size:
                continue
            elf = d[pos + off:pos + off + size]
            shoff, = struct.unpack_from("<Q", elf, 0x28)
            entry, count = struct.unpack_from("<HH", elf, 0x3a)
            for i in range(count):
                sh = shoff + i * entry
                if struct.unpack_from("<I", elf, sh + 4)[0] != SHT_NOTE:
                    continue
                o, = struct.unpack_from("<Q", elf, sh + 0x18)
                name_size, desc_size, _ = struct.unpack_from("<III", elf, o)
                at = o + 12 + (name_size + 3) // 4 * 4
                for k in msgpack.unpackb(elf[at:at + desc_size])["amdhsa.kernels"]:
                    out[k[".name"]] = k
        pos = d.find(MAGIC, pos + len(MAGIC))
    return out


@pytest.mark.parametrize("kernel,count,waves", [("copy_plan_persistent_kernel", 4, 5), ("differ_plan_kernel", 2, 8)])
def test_waves_per_simd(kernel, count, waves):
    if not os.path.exists(build.LIB):
        pytest.skip("the library is not built")
    ks = [k for n, k in _kernels(build.LIB).items() if kernel in n]
    assert len(ks) == count
    for k in ks:
        held = (k[".vgpr_count"] + 7) // 8 * 8   # allocated in eights
        assert min(8, 512 // held) >= waves, (kernel, k[".vgpr_count"])
        assert k[".private_segment_fixed_size"] == 0 and k[".vgpr_spill_count"] == 0, kernel
