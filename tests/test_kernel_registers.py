"""Register spills of the occlusion kernels, from the metadata of the built
library (CPU only)."""
import os
import re
import struct
import subprocess

import pytest

READELF = "/opt/rocm/llvm/bin/llvm-readelf"
OBJCOPY = "/opt/rocm/llvm/bin/llvm-objcopy"


def _code_objects(fat):
    """gfx950 code objects of the offload bundles in a .hip_fatbin section."""
    for m in re.finditer(b"__CLANG_OFFLOAD_BUNDLE__", fat):
        p = m.end()
        n, = struct.unpack_from("<Q", fat, p)
        p += 8
        for _ in range(n):
            off, size, k = struct.unpack_from("<QQQ", fat, p)
            triple = fat[p + 24:p + 24 + k].decode()
            p += 24 + k
            if triple.endswith("gfx950") and size:
                yield fat[m.start() + off:m.start() + off + size]


def _spills(fd, tmp_path):
    """kernel symbol -> spilled vector registers"""
    sec = tmp_path / "fatbin"
    subprocess.run([OBJCOPY, f"--dump-section=.hip_fatbin={sec}", fd.LIB_PATH, str(tmp_path / "copy.so")], check=True)
    out = {}
    for k, co in enumerate(_code_objects(sec.read_bytes())):
        path = tmp_path / f"{k}.co"
        path.write_bytes(co)
        name = None
        for line in subprocess.run([READELF, "--notes", str(path)], capture_output=True, text=True, check=True).stdout.splitlines():
            m = re.match(r"\s+\.(name|vgpr_spill_count):\s+(\S+)", line)
            if m and m.group(1) == "name" and m.group(2).startswith("_Z"):
                name = m.group(2)
            elif m and m.group(1) == "vgpr_spill_count":
                out[name] = int(m.group(2))
    return out


@pytest.mark.skipif(not os.path.exists(READELF), reason="needs llvm-readelf")
def test_batched_occlusion_spills_like_the_single_one(fd, tmp_path):
    """The batched kernels differ from the single-frame ones by where their
    arguments come from: a few registers of the allocator's choice apart (held in
    vector registers, an instance's arguments cost 30 more)."""
    fd.lib()
    s = _spills(fd, tmp_path)
    for t in "jm":   # uint32_t, uint64_t rows
        for waves in (2, 4, 8):
            one = [v for k, v in s.items() if f"k_occludeI{t}Lb0ELi{waves}E" in k]
            many = [v for k, v in s.items() if f"kb_occludeI{t}Li{waves}E" in k]
            assert len(one) == len(many) == 1, sorted(s)
            assert many[0] <= one[0] + 8, (t, waves, many, one)
