"""The tiled kernels beyond the HLLC step that test_tile_gpu.py covers, against
the one-thread-per-cell kernels on the same meshes, bit for bit (NaNs in the
same places): the HLL and Rusanov MUSCL steps and the first-order steps, at the
edges of a tile (62 cells by 2, 6, 10 or 14 rows) and on every kind of side;
the shape that the library picks for a mesh's size; states with NaN, infinite
and vacuum cells; and what a state upload leaves of the last step's gradients.
"""
import numpy as np
import pytest

from test_tile_gpu import assert_same, quadrants

pytestmark = pytest.mark.gpu

GAMMA = 1.4
SIDES = [(2, 2, 2, 2), (1, 1, 1, 1), (3, 3, 3, 3), (3, 2, 1, 3), (2, 3, 3, 1)]


def pair(zfv, nx, ny, bounds, acc, flux, limiter="MC", shape=None):
    out = []
    for tiled in (False, True):
        ctx = zfv.Context()
        ctx.mesh_rectangle(nx, ny, bounds=bounds)
        ctx.configure(acc=acc, flux=flux, limiter=limiter, cfl=0.5, gamma=GAMMA)
        if not tiled:
            for stage in range(3):
                ctx.set_launch(stage, zfv.CELL, 256)
        elif shape:
            ctx.set_launch(1, zfv.TILE, shape)
        ctx.set_state(*quadrants(nx, ny, 11))
        out.append(ctx)
    return out


def equal(a, b, what):
    for k, (x, y) in enumerate(zip(a, b)):
        assert np.array_equal(x, y, equal_nan=True), f"{what}: component {k}"


def steps_equal(ref, til, steps, what):
    for k in range(steps):
        ref.step(1)
        til.step(1)
        assert ref.dt() == til.dt(), f"{what}: dt of step {k}"
        assert_same(ref.state(), til.state(), f"{what}: step {k}")
        assert np.array_equal(ref.wait(), til.wait()), what


@pytest.mark.parametrize("acc,flux", [(1, "hllc"), (1, "hll"), (1, "rusanov"), (2, "hll"), (2, "rusanov")])
@pytest.mark.parametrize("bounds", SIDES)
@pytest.mark.parametrize("nx,ny", [(1, 1), (2, 62), (3, 63), (7, 125), (33, 64)])
def test_tiled_equals_cell_kernels(zfv, acc, flux, bounds, nx, ny):
    ref, til = pair(zfv, nx, ny, bounds, acc, flux)
    steps_equal(ref, til, 3, f"{acc} {flux} {bounds} {nx}x{ny}")


@pytest.mark.parametrize("acc", [1, 2])
@pytest.mark.parametrize("nx,ny", [(40, 40), (200, 200), (330, 280), (450, 420), (520, 390), (700, 900)])
def test_every_default_shape(zfv, acc, nx, ny):
    ref, til = pair(zfv, nx, ny, (2, 1, 3, 3), acc, "hllc")
    steps_equal(ref, til, 2, f"{acc} {nx}x{ny}")


def test_default_shapes_are_all_four(zfv):
    shapes = {nx: pair(zfv, nx, ny, (2, 1, 3, 3), 2, "hllc")[1].launch(1)
              for nx, ny in ((40, 40), (200, 200), (330, 280), (450, 420))}
    assert shapes == {40: (zfv.TILE, 256), 200: (zfv.TILE, 512), 330: (zfv.TILE, 768), 450: (zfv.TILE, 1024)}


@pytest.mark.parametrize("acc", [1, 2])
@pytest.mark.parametrize("flux", ["hllc", "hll", "rusanov"])
@pytest.mark.parametrize("limiter", ["MC", "minmod", "vanLeer"])
@pytest.mark.parametrize("value", [np.nan, np.inf, -np.inf, 0.0, 1e-310, 1e300])
def test_cells_that_are_no_state(zfv, acc, flux, limiter, value):
    """One field of a few cells out of any range (a NaN wave speed on one side
    of a face, an empty cell, overflow in the gradient), inside, at a tile's
    edge and at a wall.  Two steps: the second sees what the first left."""
    nx, ny = 19, 70
    for field in range(4):
        ref, til = pair(zfv, nx, ny, (1, 2, 1, 2), acc, flux, limiter)
        st = [a.copy() for a in quadrants(nx, ny, 5)]
        for cell in (5 * ny + 20, 6 * ny + 61, 18 * ny + 69, 0):
            st[field][cell] = value
        for k in range(2):
            got = []
            for ctx in (ref, til):
                if k == 0:
                    ctx.set_state(*st)
                ctx.step(1)
                code = 0
                try:
                    ctx.synchronize()
                except zfv.ZfvError as e:
                    code = str(e)
                out = [np.zeros(nx * ny) for _ in range(5)]
                zfv.lib().zfv_state_download(ctx.h, *[zfv._ptr(a) for a in out])   # reports the sticky error too
                got.append((code, out, ctx.wait()))
            assert got[0][0] == got[1][0]
            equal(got[0][1], got[1][1], f"field {field} step {k}")
            assert np.array_equal(got[0][2], got[1][2])


def test_upload_keeps_the_last_steps_gradients(zfv):
    """grad() after an upload is that of the last step, with the limiter the
    step had, whatever is configured or stepped in between."""
    for after in ("nothing", "limiter", "first order"):
        ref, til = pair(zfv, 30, 70, (2, 2, 2, 2), 2, "hllc")
        for ctx in (ref, til):
            ctx.step(3)
            ctx.set_state(*quadrants(30, 70, 12))
            if after == "limiter":
                ctx.configure(acc=2, flux="hllc", limiter="minmod", cfl=0.5, gamma=GAMMA)
            elif after == "first order":
                ctx.configure(acc=1, flux="hllc", limiter="MC", cfl=0.5, gamma=GAMMA)
                ctx.step(2)
        assert_same(ref.grad(), til.grad(), after)


@pytest.mark.parametrize("flux", ["hllc", "hll", "rusanov"])
@pytest.mark.parametrize("upload", [False, True])
@pytest.mark.parametrize("graphs", [False, True])
@pytest.mark.parametrize("then", ["limiter", "first order", "autotune", "first-order autotune", "refine"])
def test_gradients_are_the_last_muscl_steps(zfv, flux, upload, graphs, then):
    """grad() returns what the stage kernels stored in the last MUSCL step,
    whatever is configured, stepped, timed or adapted before it is asked for."""
    out = []
    for ctx in pair(zfv, 30, 70, (2, 1, 3, 3), 2, flux):
        ctx.graph_enable(graphs)
        ctx.step(9)   # with graphs a replay of six steps and three more
        if graphs:
            ctx.step(6)   # a replay is the last
        if upload:
            ctx.set_state(*quadrants(30, 70, 12))
        if then == "limiter":
            ctx.configure(acc=2, flux=flux, limiter="minmod", cfl=0.5, gamma=GAMMA)
        elif then == "first order":
            ctx.configure(acc=1, flux=flux, limiter="MC", cfl=0.5, gamma=GAMMA)
            ctx.step(7)
        elif then == "autotune":   # its timed launches leave the gradients of the current state
            ctx.autotune(reps=1)
        elif then == "first-order autotune":
            ctx.configure(acc=1, flux=flux, limiter="MC", cfl=0.5, gamma=GAMMA)
            ctx.autotune(reps=1)
        else:   # the slope distributor reads them
            ctx.configure(acc=2, flux=flux, limiter="vanLeer", cfl=0.5, gamma=GAMMA)
            ctx.set_flags_array(np.where(np.arange(30 * 70) % 17 < 4, 1, 0))
            ctx.refine(1, slope=True)
        out.append(ctx.state() if then == "refine" else ctx.grad())
    equal(out[0], out[1], then)


def test_gradients_after_graph_replays_and_batch_uploads(zfv):
    sizes = [(20, 33), (7, 62), (3, 3)]
    out = []
    for tiled in (False, True):
        ctx = zfv.Context()
        ctx.batch_rectangles(sizes)
        ctx.configure(acc=2, flux="hllc", limiter="MC", cfl=0.5, gamma=GAMMA)
        if not tiled:
            ctx.set_launch(1, zfv.CELL, 256)
        ctx.graph_enable(True)
        begin, count = ctx.batch_layout()
        got = []
        for seed in (1, 2, 3):
            full = [np.full(ctx.n, 3.0 + k) for k in range(5)]
            for p, (nx, ny) in enumerate(sizes):
                for k, a in enumerate(quadrants(nx, ny, seed + p)):
                    full[k][begin[p]:begin[p] + count[p]] = a
            ctx.set_state(*full)
            for n in (7, 6):
                ctx.step(n)
                got.append(ctx.state() + list(ctx.grad()))
        out.append(got)
    for a, b in zip(*out):
        assert_same(a[:5], b[:5], "states, padding cells among them")
        used = np.concatenate([np.arange(p, p + c) for p, c in zip(begin, count)])
        assert_same([g[:, used] for g in a[5:]], [g[:, used] for g in b[5:]], "gradients")


def test_device_copies_of_any_alignment(zfv):
    """State up and down through device pointers, odd sizes and rows that do
    not start on 16 bytes."""
    import ctypes as C
    hip = zfv.lib()   # the HIP runtime that the library itself is linked to
    for nx, ny, shift in ((9, 7, 0), (8, 8, 0), (8, 8, 1), (64, 33, 1)):
        n = nx * ny
        ctx = zfv.Context()
        ctx.mesh_rectangle(nx, ny)
        ctx.configure(acc=2, flux="hllc", limiter="MC", cfl=0.5, gamma=GAMMA)
        st = np.stack(quadrants(nx, ny, 3))
        host = np.zeros((5, n + 3))
        host[:, shift:shift + n] = st
        bufs = [C.c_void_p() for _ in range(2)]
        for b, h in zip(bufs, (host, np.zeros_like(host))):
            assert hip.hipMalloc(C.byref(b), C.c_size_t(host.nbytes)) == 0
            assert hip.hipMemcpy(b, C.c_void_p(h.ctypes.data), C.c_size_t(h.nbytes), 1) == 0
        at = lambda b: [b.value + 8 * ((n + 3) * k + shift) for k in range(5)]   # noqa: E731
        for _ in range(2):
            ctx.set_state_device(at(bufs[0]))
            assert zfv.lib().zfv_state_download_device(ctx.h, *[C.c_void_p(p) for p in at(bufs[1])]) == 0
            back = np.ones_like(host)
            assert hip.hipMemcpy(C.c_void_p(back.ctypes.data), bufs[1], C.c_size_t(back.nbytes), 2) == 0
            assert np.array_equal(back, host)
            dt = ctx.compute_dt()
            ctx.step(2)
            assert ctx.dt() > 0.0 and dt > 0.0
        ctx.close()
        for b in bufs:
            assert hip.hipFree(b) == 0
