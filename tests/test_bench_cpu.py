"""What bench.py takes for granted about the kernels: the tile shapes, and the
sources whose hash says whether recorded counters are those of the code that
runs."""
import os
import re
import shutil

import pytest

import bench

CSRC = os.path.join(bench.HERE, "zephyr_amd", "csrc")

# the files that hold or are included by the kernels timed under each name
SOURCES = {
    "tile": ("zfv_tile.hip", "zfv_tile_flux.hip", "zfv_tile.hpp", "zfv_pair.hpp", "zfv_physics.hpp",
             "zfv_step_common.hpp", "zfv_internal.hpp"),
    "flux1": ("zfv_kernels.hip", "zfv_tile.hip", "zfv_tile.hpp", "zfv_pair.hpp", "zfv_physics.hpp"),
    "corr": ("zfv_kernels.hip", "zfv_physics.hpp", "zfv_step_faces.hpp"),
    "grad_pred": ("zfv_kernels.hip", "zfv_step_common.hpp"),
    "k3_corr": ("zfv_3d.hip", "zfv_3d.hpp", "zfv_physics.hpp"),
}


def test_tile_shapes():
    src = open(os.path.join(CSRC, "zfv_internal.hpp")).read()
    rows = [int(v) for v in re.search(r"kTileRows\[kTileVariants\] = \{([^}]*)\}", src).group(1).split(",")]
    assert bench.TILE_ROWS == {(r + 2) * 64: r for r in rows}
    assert all(bench.tile_fused_bytes_per_cell(t) > 100.0 for t in bench.TILE_ROWS)


@pytest.mark.parametrize("kernel,name", [(k, f) for k, fs in SOURCES.items() for f in fs])
def test_source_hash_covers_the_kernels_files(tmp_path, monkeypatch, kernel, name):
    d = tmp_path / "zephyr_amd" / "csrc"
    shutil.copytree(CSRC, d)
    monkeypatch.setattr(bench, "HERE", str(tmp_path))
    before = bench.kernel_sources_sha(kernel)
    with open(d / name, "a") as f:
        f.write("// changed\n")
    assert bench.kernel_sources_sha(kernel) != before
