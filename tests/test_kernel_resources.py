"""CPU checks of what the compiler made of the kernels: registers, scratch and LDS from the code object's own metadata, against
what the host's tiling counts on."""
import os
import re
import struct

import msgpack
import pytest

from gnnhwc import _cabi

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "channels-last-groupnorm_amd", "csrc")
LDS_PER_CU = 160 * 1024
TYPES = {"DF16_": "f16", "NS_6bf16_tE": "bf16", "f": "f32", "d": "f64"}


def _kernels():
    """{mangled name: metadata} of the gfx950 code objects in the library."""
    blob = open(os.path.join(CSRC, "libgnnhwc_hip.so"), "rb").read()
    found = {}
    for bundle in re.finditer(b"__CLANG_OFFLOAD_BUNDLE__", blob):
        base = bundle.start()
        pos = base + 32
        for _ in range(struct.unpack_from("<Q", blob, base + 24)[0]):
            offset, size, length = struct.unpack_from("<QQQ", blob, pos)
            target = blob[pos + 24:pos + 24 + length]
            pos += 24 + length
            if not size or not target.endswith(b"gfx950"):
                continue
            elf = blob[base + offset:base + offset + size]
            table, = struct.unpack_from("<Q", elf, 32)
            entry, count = struct.unpack_from("<HH", elf, 54)
            for i in range(count):
                kind, _, at, _, _, length_, _, _ = struct.unpack_from("<IIQQQQQQ", elf, table + i * entry)
                end = at + length_
                while kind == 4 and at < end:  # PT_NOTE
                    name, desc, note = struct.unpack_from("<III", elf, at)
                    at += 12 + (name + 3) // 4 * 4
                    if note == 32:  # NT_AMDGPU_METADATA
                        for k in msgpack.unpackb(elf[at:at + desc], strict_map_key=False)["amdhsa.kernels"]:
                            found[k[".name"]] = k
                    at += (desc + 3) // 4 * 4
    return found


@pytest.fixture(scope="module")
def kernels():
    assert _cabi.lib is not None
    return _kernels()


def _workgroups_per_cu(k):
    """256 threads are one wavefront on each SIMD of a CU, which has 512 registers per lane, handed out by eights."""
    by_registers = 512 // ((k[".vgpr_count"] + 7) // 8 * 8)
    lds = k[".group_segment_fixed_size"]
    return min(8, by_registers, LDS_PER_CU // lds if lds else 8)


def test_the_tiling_of_the_streaming_producers_is_resident_in_one_wave(kernels):
    """The passes that leave partial results are cut into kTargetBlocks workgroups, which is one wave of resident workgroups
    only if as many of them fit a CU: with fewer, the rest start when the first are done, on a device that empties.  (The
    backward's pass over float64 data, 169 registers, is not held to it.)"""
    plan = open(os.path.join(CSRC, "gn_plan.h")).read()
    target, cus = (int(re.search(r"constexpr int %s = (\d+);" % n, plan).group(1)) for n in ("kTargetBlocks", "kNumCU"))
    seen = set()
    for name, k in kernels.items():
        m = re.match(r"_ZN2gn(?:12stats|17bwd_reduce)_kernelI(DF16_|NS_6bf16_tE|f|d)", name)
        if not m or ("bwd_reduce" in name and m.group(1) == "d"):
            continue
        seen.add(("bwd" if "bwd" in name else "fwd", TYPES[m.group(1)]))
        assert _workgroups_per_cu(k) * cus >= target, (name, k[".vgpr_count"], k[".group_segment_fixed_size"])
        assert k[".vgpr_spill_count"] == 0 and k[".private_segment_fixed_size"] == 0, name
    assert len(seen) == 7, seen
