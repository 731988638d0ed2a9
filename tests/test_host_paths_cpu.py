"""Host paths of libzfv.so that must hold when a call fails or is handed short
buffers, on the CPU: libzfv.so over a stand-in for the HIP runtime
(tests/hostshim/hip_stub.cpp), which checks copies against the allocations,
records the launches without running them, and makes chosen calls fail."""
import os
import shutil
import subprocess
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PRELUDE = """
import ctypes as C, sys
import numpy as np
hip = C.CDLL(sys.argv[1], C.RTLD_GLOBAL)
hip.stub_launch.restype = C.c_char_p
hip.stub_word.restype = C.c_uint64
hip.stub_pinned.restype = C.c_size_t
import zephyr_amd as Z

def launches():
    return [(hip.stub_launch(i).decode(), hip.stub_word(i)) for i in range(hip.stub_launches())]

def fails(call):
    try:
        call()
    except Z.ZfvError:
        return True
    return False
"""


@pytest.fixture(scope="module")
def stub(tmp_path_factory):
    if shutil.which("g++") is None or not os.path.exists("/opt/rocm/include/hip/hip_runtime_api.h"):
        pytest.skip("needs g++ and the HIP headers")
    so = str(tmp_path_factory.mktemp("stub") / "libhipstub.so")
    subprocess.run(["g++", "-O1", "-std=c++17", "-shared", "-fPIC", "-w", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                    os.path.join(ROOT, "tests", "hostshim", "hip_stub.cpp"), "-o", so], check=True)

    def run(code):
        out = subprocess.run([sys.executable, "-c", PRELUDE + code, so], capture_output=True, text=True, cwd=ROOT,
                             timeout=120)
        assert out.returncode == 0, out.stdout + out.stderr
    return run


@pytest.mark.parametrize("overlap,call,after", [
    (0, "8k_mm_crpI", 0), (0, "10k_mm_flux1I", 0), (1, "10k_mm_flux1I", 0), (2, "8k_mm_crpI", 0),
    (2, "hipStreamWaitEvent", 1), (2, "hipStreamWaitEvent", 2), (2, "15k_mm_take_count", 0)])
def test_composite_face_counters_are_clear_after_a_failed_step(stub, overlap, call, after):
    """Every marking starts from counters that nothing has appended to: taken
    by the last step's update, or cleared after a step that failed between."""
    stub(f"""
ctx = Z.Context()
ctx.mesh_rectangle(8, 8)
ctx.mm_configure([(1.4, 0, 0, 718.0, 0, 1.2), (1.6, 0, 0, 3116.0, 0, 0.2)])
ctx.mm_set_overlap({overlap})
one = np.ones(64)
ctx.mm_set_state(one, one, one, one, np.stack([one, 0 * one]))
hip.stub_keep(b"10k_fill_u64", 0)
hip.stub_keep(b"13k_mm_crp_markI", 8)
ctx.mm_step(1)
hip.stub_reset()
ctx.mm_step(1)
calls = launches()
count = [w for name, w in calls if "k_mm_crp_mark" in name]
assert len(count) == 1 and not any("k_fill_u64" in name for name, w in calls), calls   # the update takes them
for attempt in range(2):
    hip.stub_fail({call.encode()!r}, {after})
    assert fails(lambda: ctx.mm_step(1))
    hip.stub_reset()
    if attempt:
        ctx.mm_step(1)
        calls = launches()
        mark = [i for i, (name, w) in enumerate(calls) if "k_mm_crp_mark" in name][0]
        assert any("k_fill_u64" in name and w == count[0] for name, w in calls[:mark]), calls
hip.stub_reset()
ctx.mm_step(1)
assert not any("k_fill_u64" in name for name, w in launches())
""")


@pytest.mark.parametrize("row", range(5))
@pytest.mark.parametrize("short", [8, 8 * 35])
def test_short_device_rows_are_refused(stub, row, short):
    """A device row that ends before its last cell is refused, as by hipMemcpy,
    and no kernel is given it; a row of exactly the mesh's cells, at the end of a
    larger allocation, is copied by the kernel, one off an 8-byte boundary is not."""
    stub(f"""
n = 36
ctx = Z.Context()
ctx.mesh_rectangle(6, 6)
ctx.configure()
one = np.ones(n)
ctx.set_state(one, one, one, one, one)

def device(nbytes):
    p = C.c_void_p()
    assert hip.hipMalloc(C.byref(p), C.c_size_t(nbytes)) == 0
    return p.value

up, down = Z.lib().zfv_state_upload_device, Z.lib().zfv_state_download_device

def go(call, rows):
    hip.stub_reset()
    code = call(ctx.h, *[C.c_void_p(p) for p in rows])
    return code, any("k_state_copy" in name for name, w in launches())

rows = [device(8 * n) for _ in range(5)]
tail = device(8 * n + 16)
for call in (up, down):
    assert go(call, rows) == (0, True)
    end = list(rows)
    end[{row}] = tail + 16
    assert go(call, end) == (0, True)
    off = list(rows)
    off[{row}] = tail + 4
    assert go(call, off) == (0, False)
    late = list(rows)
    late[{row}] = tail + 24
    code, kernel = go(call, late)
    assert code == Z.ZFV_ERR_HIP and not kernel
    less = list(rows)
    less[{row}] = device(8 * n - {short})
    code, kernel = go(call, less)
    assert code == Z.ZFV_ERR_HIP and not kernel
    one = device(8 * 5 * n)   # the rows of one allocation, and of one that ends in the last row
    assert go(call, [one + 8 * n * k for k in range(5)]) == (0, True)
    one = device(8 * 5 * n - {short})
    code, kernel = go(call, [one + 8 * n * k for k in range(5)])
    assert code == Z.ZFV_ERR_HIP and not kernel
""")


@pytest.mark.parametrize("rows,block", [(2, 256), (6, 512), (10, 768), (14, 1024)])
def test_tile_shape_that_runs_is_reported_kept_and_tuned(stub, rows, block):
    """launch() reports the shape the steps run, set_launch(1, TILE, 0) and
    set_launch of what was reported keep it, and the autotuner takes the
    fastest of all four."""
    stub(f"""
def make(nx, ny):
    ctx = Z.Context()
    ctx.mesh_rectangle(nx, ny)
    ctx.configure(acc=2, flux="hllc", limiter="MC")
    one = np.ones(nx * ny)
    ctx.set_state(one, one, one, one, one)
    return ctx

def runs(ctx):
    hip.stub_reset()
    ctx.step(1)
    name = [n for n, w in launches() if "k_tile_step" in n][-1]
    return (int(name.split("ELi")[3].split("E")[0]) + 2) * 64

seen = set()
for nx, ny in ((8, 8), (64, 48), (200, 200), (330, 280), (520, 390), (900, 700)):
    ctx = make(nx, ny)
    shape = runs(ctx)
    seen.add(shape)
    assert ctx.launch(1) == (Z.TILE, shape), (nx, ny, ctx.launch(1), shape)
    ctx.set_launch(1, Z.TILE, 0)
    assert runs(ctx) == shape and ctx.launch(1) == (Z.TILE, shape)
    ctx.set_launch(1, Z.TILE, {block})
    assert runs(ctx) == {block} and ctx.launch(1) == (Z.TILE, {block})
assert 256 in seen and len(seen) > 1, seen
ctx = make(64, 48)
hip.stub_cost(b"k_tile_stepILi3ELi3E", C.c_double(0.5))
hip.stub_cost(b"k_tile_stepILi3ELi3ELi{(6, 10, 14, 2).index(rows)}ELi{rows}E", C.c_double(0.25))
ms = ctx.autotune(reps=2)
assert ctx.launch(1) == (Z.TILE, {block}) and runs(ctx) == {block}
assert np.all(ms[1, 3] == [0.25 if r == {rows} else 0.5 for r in (6, 10, 14)]), ms[1, 3]
""")


@pytest.mark.parametrize("flux", ["hllc", "hll", "rusanov"])
def test_narrow_meshes_run_the_cell_kernels(stub, flux):
    """The tiled steps run where they take less than one thread per cell: not on
    meshes of a few cells along j, whose tiles are mostly lanes without a cell; a
    caller's choice stands."""
    stub(f"""
def runs(ctx):
    hip.stub_reset()
    ctx.step(1)
    return any("k_tile" in n for n, w in launches())

for acc in (1, 2):
    for nx, ny, tiled in ((10000, 1, False), (100000, 1, False), (50000, 4, False), (20000, 10, False), (5000, 4, False),
                          (1, 1, True), (2, 62, True), (3, 63, True), (7, 125, True), (33, 64, True), (19, 70, True),
                          (8, 8, True), (1, 1000, True), (64, 48, True), (4, 5000, True), (300, 200, True),
                          (900, 700, True)):
        ctx = Z.Context()
        ctx.mesh_rectangle(nx, ny)
        ctx.configure(acc=acc, flux={flux!r}, limiter="MC")
        one = np.ones(nx * ny)
        ctx.set_state(one, one, one, one, one)
        assert runs(ctx) == tiled, (acc, nx, ny)
        if acc == 2:
            assert (ctx.launch(1)[0] == Z.TILE) == tiled
            ctx.set_launch(1, Z.TILE, 0)
            assert runs(ctx) and ctx.launch(1)[0] == Z.TILE
            ctx.set_launch(1, Z.CELL, 256)
        else:
            ctx.set_launch(0, Z.CELL, 256)
        assert not runs(ctx)
""")


def test_tile_tables_of_a_mesh_are_three_copies(stub):
    """A Rectangle's mesh upload copies its tile tables (problems, columns, rows)
    in one copy each, beside the 22 of the mesh arrays."""
    stub("""
ctx = Z.Context()
before = hip.stub_copies()
ctx.mesh_rectangle(5, 7)
assert hip.stub_copies() - before == 25, hip.stub_copies() - before
""")


def test_3d_transfers_hold_little_pinned_memory(stub):
    """A 3D context holds the pinned memory its largest transfer needs, at most two
    parts of 2 MiB, until it is closed; without pinned memory or events the
    arrays are copied as they are."""
    stub("""
base = hip.stub_pinned()

def make(n):
    ctx = Z.Context3()
    ctx.mesh_cuboid(1, 1, n)
    ctx.configure()
    one = np.ones(n)
    return ctx, lambda: ctx.set_state(one, one, one, one, one, one)

ctx, up = make(1)
up()
ctx.state()
assert hip.stub_pinned() - base == 48, hip.stub_pinned() - base
ctx.grad()
assert hip.stub_pinned() - base == 120
ctx.close()
assert hip.stub_pinned() == base
ctx, up = make(200000)
up()
ctx.state()
ctx.grad()
assert hip.stub_pinned() - base <= 4 << 20
ctx.close()
assert hip.stub_pinned() == base
for call in ("hipHostMalloc", "hipEventCreate"):
    ctx, up = make(50000)
    for transfer in (up, ctx.state, ctx.grad):
        hip.stub_fail(call.encode(), 0)
        before = hip.stub_copies()
        transfer()
        if transfer is up:   # one that failed to have it copies, the next has it
            assert hip.stub_copies() - before >= 6
    ctx.close()
assert hip.stub_pinned() == base
""")
