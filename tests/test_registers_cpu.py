"""Spilled registers of the 3D corrector as it was compiled: a bound on the waves
a SIMD that suits one flux can make another spill by the hundred (HLL 133 ->
250 us at 96^3 cells) and still give the right results."""
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


@pytest.mark.skipif(not os.path.exists(READELF), reason="needs llvm-readelf")
def test_3d_corrector_spills_few_registers(zfv, tmp_path):
    spills = {}
    for i, obj in enumerate(code_objects(zfv.LIB_PATH)):
        f = tmp_path / f"{i}.o"
        f.write_bytes(obj)
        if b"k3_corr" not in obj:
            continue
        notes = subprocess.run([READELF, "--notes", str(f)], capture_output=True, text=True, check=True).stdout
        name = None
        for line in notes.splitlines():
            m = re.match(r"\s+\.name:\s+(\S*k3_corr\S*)", line)
            name = m.group(1) if m else (None if re.match(r"\s+\.name:\s+_Z", line) else name)
            m = re.match(r"\s+\.vgpr_spill_count:\s+(\d+)", line)
            if m and name:
                spills[name] = int(m.group(1))
    assert len(spills) == 16, spills   # eight fluxes, tables and slot arrays
    assert max(spills.values()) <= 16, spills
