"""The force kernels keep LDS addresses in mask words of 12 bits (k_force,
kMaxStaged) and lists of 16 (k_force_split): right only while k_force has no
static LDS before its dynamic one, and k_force_split no more than its plan
counts on (kStaticLds).  Read from the metadata of the built library's kernels."""
from __future__ import annotations

import os
import re
import struct

import msgpack

from particle_life import _native

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "particle-life-app_amd", "csrc")


def _kernels():
    """Metadata of every gfx950 kernel: the code objects of the offload bundles
    in the library, their AMDGPU metadata notes (msgpack)."""
    blob = open(_native.LIB_PATH, "rb").read()
    got = []
    for m in re.finditer(b"__CLANG_OFFLOAD_BUNDLE__", blob):
        at = m.end()
        count, = struct.unpack_from("<Q", blob, at)
        at += 8
        for _ in range(count):
            off, size, tlen = struct.unpack_from("<QQQ", blob, at)
            triple = blob[at + 24:at + 24 + tlen]
            at += 24 + tlen
            if b"gfx950" not in triple:
                continue
            elf = blob[m.start() + off:m.start() + off + size]
            shoff, = struct.unpack_from("<Q", elf, 0x28)
            entsize, num = struct.unpack_from("<HH", elf, 0x3A)
            for k in range(num):
                kind, _, _, o, n = struct.unpack_from("<IQQQQ", elf, shoff + k * entsize + 4)
                if kind != 7:                                   # SHT_NOTE
                    continue
                namesz, descsz, _ = struct.unpack_from("<III", elf, o)
                desc = o + 12 + (namesz + 3 & ~3)
                got += msgpack.unpackb(elf[desc:desc + descsz])["amdhsa.kernels"]
    return {k[".name"]: k for k in got}


def test_static_lds_of_the_force_kernels():
    src = open(os.path.join(CSRC, "plife.hip")).read()
    static = int(re.search(r"kStaticLds = (\d+)", src).group(1))
    kernels = _kernels()
    staged = {n: k for n, k in kernels.items() if re.search(r"7k_forceI", n)}
    split = {n: k for n, k in kernels.items() if "13k_force_splitI" in n}
    assert len(staged) == 48 and len(split) == 16
    for n, k in staged.items():
        assert k[".group_segment_fixed_size"] == 0, n
    for n, k in split.items():
        assert k[".group_segment_fixed_size"] <= static, n
    # and neither spills, which their occupancy is planned without
    for n, k in {**staged, **split}.items():
        assert k[".vgpr_spill_count"] == 0 and k[".private_segment_fixed_size"] == 0, n
