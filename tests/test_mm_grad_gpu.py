"""The multi-material gradient's chunks of components beside each other (small
meshes) and in turn (large ones).  With cells of 1/256 every coordinate is exact,
so a periodic mesh repeated three times along y has the same stencils cell by
cell, lies on the other side of the line (65536 and 196608 cells), and gives the
same gradients and states bit for bit."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SIDE = 256
# gases: (gamma, P0, e0, Cv, T0, rho_ref)
GASES = [(1.4, 0.0, 0.0, 718.0, 0.0, 1.25), (1.67, 0.0, 0.0, 3116.0, 0.0, 0.18), (1.3, 0.0, 0.0, 655.0, 0.0, 1.98),
         (1.2, 0.0, 0.0, 900.0, 0.0, 1.5)]


@pytest.mark.parametrize("mats", [1, 2, 3, 4])
@pytest.mark.parametrize("limiter", [2, 3])
def test_gradient_chunks_beside_and_in_turn(zfv, mats, limiter):
    rng = np.random.default_rng(mats)
    material = np.kron(rng.integers(0, mats, size=(16, 16)), np.ones((16, 16), int))
    # uniform along the edges: the reference extrapolates a periodic neighbour from its own centre
    inside = np.zeros((SIDE, SIDE))
    inside[6:-6, 6:-6] = 1.0
    material = np.where(inside > 0.0, material, 0)
    beta = np.stack([(material == i).astype(float) for i in range(mats)])
    beta[:, 40, 8:-8] = 1.0 / mats       # a mixed row
    rho = 1.0 + 0.1 * inside * rng.random((SIDE, SIDE))
    u, v = 10.0 * inside * rng.normal(size=(2, SIDE, SIDE))
    P = 1.0e5 * (1.0 + 0.1 * inside * rng.random((SIDE, SIDE)))
    out = []
    for k in (1, 3):
        ctx = zfv.Context()
        ctx.mesh_rectangle(SIDE, k * SIDE, ymax=float(k), bounds=(zfv.PERIODIC,) * 4)
        ctx.mm_configure(GASES[:mats], 0.4)
        ctx.mm_set_accuracy(2)
        ctx.mm_set_limiter(limiter)

        def rep(a):
            return np.ascontiguousarray(np.concatenate([a] * k, axis=1).reshape(-1))

        ctx.mm_set_state(rep(rho), rep(u), rep(v), rep(P), np.stack([rep(b) for b in beta]))
        ctx.mm_step(1)
        z = ctx.mm_state()
        out.append([a.reshape(-1, SIDE, k * SIDE)[:, :, :SIDE] for a in (*ctx.mm_grad(), *z.values())])
        assert np.any(out[-1][0][0] != 0.0)
    for a, b in zip(*out):
        assert np.array_equal(a, b, equal_nan=True)
