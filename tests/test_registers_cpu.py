"""Registers and scratch memory of kernels as they were compiled.  A bound on the
waves a SIMD that suits one flux can make another spill by the hundred (3D
corrector, HLL 133 -> 250 us at 96^3 cells) and still give the right results; so
can an array that the compiler indexes at run time."""
import os
import re
import struct
import subprocess

import pytest

READELF = "/opt/rocm/llvm/bin/llvm-readelf"
BUNDLE = b"__CLANG_OFFLOAD_BUNDLE__"


def code_objects(path):
    """The gfx950 code objects of a library's offload bundles."""
    data = open(path, "rb").read()
    at = data.find(BUNDLE)
    while at >= 0:
        count, = struct.unpack_from("<Q", data, at + len(BUNDLE))
        p = at + len(BUNDLE) + 8
        for _ in range(count):
            off, size, n = struct.unpack_from("<QQQ", data, p)
            name = data[p + 24:p + 24 + n]
            p += 24 + n
            if name.endswith(b"gfx950") and size:
                yield data[at + off:at + off + size]
        at = data.find(BUNDLE, p)


def metadata(path, tmp_path, part, field):
    """{kernel: value} of a metadata field of the kernels whose names hold `part`."""
    out = {}
    for i, obj in enumerate(code_objects(path)):
        if part.encode() not in obj:
            continue
        f = tmp_path / f"{i}.o"
        f.write_bytes(obj)
        notes = subprocess.run([READELF, "--notes", str(f)], capture_output=True, text=True, check=True).stdout
        for kernel in re.split(r"\n\s+- \.agpr_count", notes)[1:]:
            name = re.search(r"\.name:\s+(_Z\S+)", kernel).group(1)
            if part in name:
                out[name] = int(re.search(rf"\.{field}:\s+(\d+)", kernel).group(1))
    return out


@pytest.mark.skipif(not os.path.exists(READELF), reason="needs llvm-readelf")
def test_3d_corrector_spills_few_registers(zfv, tmp_path):
    spills = metadata(zfv.LIB_PATH, tmp_path, "k3_corr", "vgpr_spill_count")
    assert len(spills) == 16, spills   # eight fluxes, tables and slot arrays
    assert max(spills.values()) <= 16, spills


@pytest.mark.skipif(not os.path.exists(READELF), reason="needs llvm-readelf")
def test_mixtures_of_any_size_stay_out_of_scratch(zfv, tmp_path):
    """The multi-material kernels choose a material by selects, not through a copy
    of the mixture in scratch memory."""
    scratch = metadata(zfv.LIB_PATH, tmp_path, "k_mm_", "private_segment_fixed_size")
    assert sum("k_mm_crpI" in k for k in scratch) == 8, scratch   # one to four materials, both orders
    assert not any(scratch.values()), {k: v for k, v in scratch.items() if v}
