"""The three-dimensional corrector's two sources of a neighbour's record (its
workgroup's LDS, memory) and the paired layouts, at the sizes where they meet:
n around a workgroup's 256 cells, rows longer than a workgroup, axes one cell
long.  Bar: value equality with the oracle, as both sides are the same sequence
of correctly rounded IEEE operations; the slot arrays in place of the tables give
the same values."""
import numpy as np
import pytest

from test_3d_gpu import LIMITERS, STATE, assert_equal, make_pair

pytestmark = pytest.mark.gpu

SHAPES = [(1, 1, 1), (1, 1, 257), (5, 3, 17), (4, 8, 8), (257, 1, 1), (3, 2, 300), (2, 130, 2), (3, 5, 64), (7, 6, 96)]


@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("bounds", [(3,) * 6, (1, 2, 2, 1, 1, 2)])
@pytest.mark.parametrize("acc", [1, 2])
def test_shapes_match_oracle(oracle, zfv, shape, bounds, acc):
    m, s, ctx = make_pair(oracle, zfv, shape, box=(-0.2, 1.1, 0.0, 0.7, 0.1, 1.3), bounds=bounds, acc=acc,
                          flux="hllc", limiter=LIMITERS.index("MC"), seed=sum(shape))
    n = m.n
    if acc == 2:   # robust faces on both sides of a workgroup's edge
        wait = np.where(np.arange(n) % 37 == 5, 2, 0).astype(np.int32)
        s.set_wait(wait)
        ctx.set_wait(wait)
    for step in range(3):
        s.update()
        ctx.step(1)
        assert_equal(ctx.state(), s.state(), STATE, f"{shape} step {step}")
        if acc == 2:
            assert np.array_equal(ctx.grad(), s.grad())
            assert np.array_equal(ctx.wait(), s.wait())


def test_tables_and_slot_arrays_agree(oracle, zfv):
    out = []
    for tables in (True, False):
        m, s, ctx = make_pair(oracle, zfv, (2, 2, 2))
        ctx.set_geometry_tables(tables)
        ctx.mesh_cuboid(9, 11, 33, 0.0, 0.9, -0.3, 1.0, 0.0, 2.0, bounds=(3, 3, 1, 2, 2, 1))
        ctx.configure(acc=2, flux="hllc", limiter="MC", cfl=0.5, gamma=1.4)
        assert ctx.geometry_tables() == tables
        rng = np.random.default_rng(5)
        r, p = 1.0 + rng.random(ctx.n), 1.0 + rng.random(ctx.n)
        u, v, w = 0.3 * rng.normal(size=(3, ctx.n))
        ctx.set_state(r, u, v, w, p)
        ctx.step(4)
        out.append(list(ctx.state()) + [ctx.grad().ravel()])
    for a, b in zip(*out):
        assert np.array_equal(a, b)
