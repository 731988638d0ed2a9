"""States and gradients of the 3D step to and from host arrays, which go through
two parts of pinned memory, at the edges of a part (43690 cells of a state,
17476 of the gradients), against the same arrays in device memory, which are
copied whole."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

STATE, GRAD = (2 << 20) // 48, (2 << 20) // 120


class Device:
    """A host array mirrored in device memory."""

    def __init__(self, hip, size):
        self.hip, self.size, self.p = hip, size, C.c_void_p()
        assert hip.hipMalloc(C.byref(self.p), C.c_size_t(8 * size)) == 0

    def put(self, a):
        assert self.hip.hipMemcpy(self.p, C.c_void_p(a.ctypes.data), C.c_size_t(8 * self.size), 1) == 0

    def get(self):
        a = np.empty(self.size)
        assert self.hip.hipMemcpy(C.c_void_p(a.ctypes.data), self.p, C.c_size_t(8 * self.size), 2) == 0
        return a

    def free(self):
        assert self.hip.hipFree(self.p) == 0


@pytest.mark.parametrize("n", [1, 7, GRAD - 1, GRAD, GRAD + 1, 2 * GRAD, 2 * GRAD + 1, STATE - 1, STATE, STATE + 1,
                               2 * STATE, 3 * STATE + 5, 300000])
def test_host_arrays_equal_device_arrays(zfv, n):
    rng = np.random.default_rng(n)
    lib = zfv.lib()
    src = [1.0 + rng.random(n), *rng.normal(size=(3, n)), 1.0 + rng.random(n), 2.0 + rng.random(n)]
    dev = [Device(lib, n) for _ in range(6)]
    dg = Device(lib, 15 * n)
    got = []
    for host in (True, False):
        ctx = zfv.Context3()
        ctx.mesh_cuboid(1, 1, n, 0.0, 1.0 / n, 0.0, 1.0 / n, 0.0, 1.0)
        ctx.configure(acc=2, flux="hllc", limiter="MC", cfl=0.4, gamma=1.4)
        for again in range(2):   # the pinned parts are reused
            if host:
                ctx.set_state(*[a + again for a in src])
                up = ctx.state()
            else:
                for d, a in zip(dev, src):
                    d.put(a + again)
                assert lib.zfv3_state_upload(ctx.h, *[d.p for d in dev]) == 0
                assert lib.zfv3_state_download(ctx.h, *[d.p for d in dev]) == 0
                up = [d.get() for d in dev]
            for a, b in zip(up, src):
                assert np.array_equal(a, b + again)
            ctx.step(2)
            if host:
                got.append(list(ctx.state()) + [ctx.grad().ravel()])
            else:
                assert lib.zfv3_state_download(ctx.h, *[d.p for d in dev]) == 0
                assert lib.zfv3_grad_download(ctx.h, dg.p) == 0
                got.append([d.get() for d in dev] + [dg.get()])
        ctx.close()
    for d in dev + [dg]:
        d.free()
    for a, b in zip(got[:2], got[2:]):
        for x, y in zip(a, b):
            assert np.array_equal(x, y)
    # fields left out stay as they are
    ctx = zfv.Context3()
    ctx.mesh_cuboid(1, 1, n)
    ctx.configure()
    ctx.set_state(*src)
    p = np.zeros(n)
    assert lib.zfv3_state_download(ctx.h, None, None, None, None, C.c_void_p(p.ctypes.data), None) == 0
    assert np.array_equal(p, src[4])
