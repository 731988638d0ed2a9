"""The work that a user of zephyr_amd has it do, as cases that can be timed.

A case is one call sequence of a simulation program on a context the program
keeps: set a state (device arrays), advance it, read the state back; or, where
the mesh follows the flow, one adaptation cycle of a running simulation.  The
meshes, schemes and data are those of the repository's own workloads and tests
(four-quadrant Riemann data, random smooth fields, blasts, shock-bubbles), over
sizes from a single small problem to the largest meshes they use.

FP64 throughout.
"""
import ctypes as C
import math

import numpy as np
import torch

import zephyr_amd as Z
from zephyr_amd import problems

GAMMA = 1.4
WALL, ZOE, PERIODIC = Z.WALL, Z.ZOE, Z.PERIODIC
BOUNDS = {"open": (ZOE,) * 4, "walls": (WALL,) * 4, "periodic": (PERIODIC,) * 4,
          "mixed": (WALL, ZOE, PERIODIC, PERIODIC)}
BOUNDS3 = {"open": (ZOE,) * 6, "walls": (WALL,) * 6, "periodic": (PERIODIC,) * 6}


def listed():
    return [
        # A control loop on a small problem: one step, then its dt, at every
        # call.  Latency and launches are what it pays for.
        dict(name="rect64x48_step_dt", kind="rect", nx=64, ny=48, acc=2, flux="hllc", limiter="MC", bounds="open",
             data="quadrants", steps=1),
        # The plain first-order step of the reference's 2D Riemann test.
        dict(name="rect200_first_order", kind="rect", nx=200, ny=200, acc=1, flux="hllc", limiter="MC",
             bounds="open", data="quadrants", steps=20),
        # The MUSCL + HLLC step of a mid-sized mesh, ragged, walls and a
        # periodic direction.
        dict(name="rect517x389_minmod", kind="rect", nx=517, ny=389, acc=2, flux="hllc", limiter="minmod",
             bounds="mixed", data="smooth", steps=16),
        # Another flux: the second-order step with HLL on a closed box.
        dict(name="rect611x450_hll", kind="rect", nx=611, ny=450, acc=2, flux="hll", limiter="vanLeer",
             bounds="walls", data="quadrants", steps=12),
        # The large uniform mesh.
        dict(name="rect1361x1023_mc", kind="rect", nx=1361, ny=1023, acc=2, flux="hllc", limiter="MC",
             bounds="open", data="smooth", steps=10),
        # Adaptive mesh: one cycle of a running simulation (flags, refine /
        # coarsen, four steps) following a bubble carried around a periodic
        # box, up to three levels.
        dict(name="amr256_cycle", kind="amr", nx=256, ny=256, max_level=3, limiter="minmod", steps=4),
        # An ensemble of independent uneven problems in one context, steps
        # replayed from graphs.
        dict(name="batch40_uneven", kind="batch", problems=40, smin=33, smax=257, limiter="MC", steps=12),
        # Gradient of a final-time functional: forward with checkpoints and
        # the reverse sweep.
        dict(name="adjoint317x290", kind="adjoint", nx=317, ny=290, limiter="MC", steps=20, every=10),
        # Two materials (water with an air bubble, a shock), first order with
        # composite Riemann fluxes.
        dict(name="mm384_first_order", kind="mm", nx=384, ny=384, acc=1, steps=60),
        # ... and second order, on a ragged mesh.
        dict(name="mm301x245_second_order", kind="mm", nx=301, ny=245, acc=2, steps=40),
        # The three-dimensional step of a running simulation, with its state
        # read back.
        dict(name="cube96_mc", kind="cube", nx=96, ny=96, nz=96, acc=2, flux="hllc", limiter="MC", bounds="walls",
             steps=24),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["rect", "rect", "rect", "amr", "batch", "adjoint", "mm", "mm", "cube", "cube"])
    if kind == "rect":
        cells = math.exp(rng.uniform(math.log(2500.0), math.log(1.3e6)))
        aspect = math.exp(rng.uniform(math.log(0.5), math.log(2.0)))
        nx = max(24, int(math.sqrt(cells * aspect)))
        ny = max(24, int(cells / nx))
        acc = rng.choice([1, 2, 2, 2])
        flux = rng.choice(["hllc", "hllc", "hllc", "hll", "rusanov"])
        return dict(kind="rect", nx=nx, ny=ny, acc=acc, flux=flux,
                    limiter=rng.choice(["MC", "minmod", "vanLeer", "Koren"]),
                    bounds=rng.choice(["open", "walls", "periodic", "mixed"]),
                    data=rng.choice(["quadrants", "smooth"]), steps=rng.choice([1, 4, 7, 10]))
    if kind == "amr":
        return dict(kind="amr", nx=_log_int(rng, 64, 256), ny=_log_int(rng, 64, 256), max_level=rng.randint(1, 3),
                    limiter=rng.choice(["minmod", "MC"]), steps=rng.randint(2, 5))
    if kind == "batch":
        return dict(kind="batch", problems=_log_int(rng, 4, 40), smin=rng.randint(17, 64), smax=rng.randint(100, 257),
                    limiter=rng.choice(["MC", "minmod"]), steps=rng.choice([6, 12]))
    if kind == "adjoint":
        return dict(kind="adjoint", nx=_log_int(rng, 40, 310), ny=_log_int(rng, 40, 290),
                    limiter=rng.choice(["MC", "minmod"]), steps=rng.randint(5, 18), every=rng.randint(3, 8))
    if kind == "mm":
        acc = rng.choice([1, 2])
        top = 380 if acc == 1 else 270
        return dict(kind="mm", nx=_log_int(rng, 48, top), ny=_log_int(rng, 48, top), acc=acc,
                    steps=rng.randint(10, 40))
    return dict(kind="cube", nx=_log_int(rng, 12, 96), ny=_log_int(rng, 12, 96), nz=_log_int(rng, 12, 95),
                acc=rng.choice([1, 2, 2, 2]), flux=rng.choice(["hllc", "hllc", "rusanov"]),
                limiter=rng.choice(["MC", "minmod"]), bounds=rng.choice(["open", "walls", "periodic"]),
                steps=rng.randint(4, 24))


# ---- inputs ------------------------------------------------------------------
def _centres(n, lo=0.0, hi=1.0):
    v = lo + ((hi - lo) * np.arange(n + 1)) / n
    return 0.5 * (v[:-1] + v[1:])


def _grid(*ns):
    return [g.reshape(-1) for g in np.meshgrid(*[_centres(n) for n in ns], indexing="ij")]


def _waves(rng, xs, modes=5):
    """A smooth random field of unit scale: a few seeded Fourier modes."""
    f = np.zeros_like(xs[0])
    for _ in range(modes):
        k = 2.0 * np.pi * rng.integers(1, 4, size=len(xs))
        f += rng.normal() * np.cos(sum(a * x for a, x in zip(k, xs)) + 2.0 * np.pi * rng.random())
    return f / math.sqrt(modes)


def _smooth2(nx, ny, seed):
    rng = np.random.default_rng(seed)
    xs = _grid(nx, ny)
    rho = 1.0 + 0.1 * _waves(rng, xs)
    p = 1.0 + 0.1 * _waves(rng, xs)
    u, v = 0.2 * _waves(rng, xs), 0.2 * _waves(rng, xs)
    return rho, u, v, p, problems.energy_rP(rho, p, GAMMA)


def _sides(case):
    return [int(n) for n in np.linspace(case["smin"], case["smax"], case["problems"])]


def _batch_state(case, seed):
    """The concatenated states (each problem from a 512-cell boundary on, ones
    between them) and each problem's side and first cell."""
    rng = np.random.default_rng(seed)
    parts, where, at = [], [], 0
    for n in _sides(case):
        pad = -(n * n) % 512
        st = np.stack(problems.four_quadrant(*_grid(n, n), int(rng.integers(1 << 30))))
        parts.append(np.concatenate([st, np.ones((5, pad))], axis=1))
        where.append((n, at))
        at += n * n + pad
    return np.concatenate(parts, axis=1), where


def _state2(case, seed):
    if case.get("data") == "quadrants":
        cx, cy = _grid(case["nx"], case["ny"])
        return problems.four_quadrant(cx, cy, seed)
    return _smooth2(case["nx"], case["ny"], seed)


def _blast3(case, seed):
    rng = np.random.default_rng(seed)
    x = _grid(case["nx"], case["ny"], case["nz"])
    c = rng.uniform(0.4, 0.6, size=3)
    r = np.sqrt(sum((a - b) ** 2 for a, b in zip(x, c)))
    rho = 1.0 + 0.5 * (r < 0.25) + 0.05 * _waves(rng, x)
    p = 1.0 + 4.0 * (r < 0.25)
    u, v, w = (0.1 * _waves(rng, x) for _ in range(3))
    return rho, u, v, w, p, p / ((GAMMA - 1.0) * rho)


def _carried(cx, cy, seed):
    """A round bubble in a uniform stream; pressure and velocity are uniform,
    so the bubble is carried through the periodic box for ever."""
    rng = np.random.default_rng(seed)
    c = rng.uniform(0.35, 0.65, size=2)
    rho = np.where((cx - c[0]) ** 2 + (cy - c[1]) ** 2 < 0.2 ** 2, 1.0, 0.1)
    a, one = rng.uniform(0.0, 2.0 * np.pi), np.ones_like(cx)
    return rho, math.cos(a) * one, math.sin(a) * one, one, problems.energy_rP(rho, one, GAMMA)


def _bubble(case, seed):
    """The water / air shock-bubble, the fluid stirred by a smooth flow
    without divergence."""
    cx, cy = _grid(case["nx"], case["ny"])
    rho, u, v, P, beta = problems.mm_bubble_shock(cx, cy, 1.0 / max(case["nx"], case["ny"]), seed)
    return rho, u + 30.0 * np.cos(2.0 * cy), v - 30.0 * np.sin(3.0 * cx), P, beta


def _on_gpu(rows):
    return torch.from_numpy(np.ascontiguousarray(np.stack(rows))).cuda()


def _adapt_cycle(ctx, case):
    ctx.set_flags(1, 0.1)
    ctx.refine(case["max_level"], slope=True)
    ctx.step(case["steps"])


def prepare(case, seed):
    kind = case["kind"]
    s = dict(case=case)
    if kind == "cube":
        ctx = Z.Context3()
        ctx.mesh_cuboid(case["nx"], case["ny"], case["nz"], bounds=BOUNDS3[case["bounds"]])
        ctx.configure(acc=case["acc"], flux=case["flux"], limiter=case["limiter"], cfl=0.5, gamma=GAMMA)
        ctx.set_state(*_blast3(case, seed))
        s["ctx"] = ctx
        return s
    ctx = Z.Context()
    s["ctx"] = ctx
    if kind == "batch":
        ctx.batch_rectangles([(n, n) for n in _sides(case)])
        st = _batch_state(case, seed)[0]
        ctx.configure(acc=2, flux="hllc", limiter=case["limiter"], cfl=0.5, gamma=GAMMA)
        ctx.graph_enable(True)
        s["in"], s["out"] = _on_gpu(st), torch.empty(5, ctx.n, dtype=torch.float64, device="cuda")
    elif kind == "mm":
        ctx.mesh_rectangle(case["nx"], case["ny"])
        ctx.mm_configure([problems.WATER, problems.AIR], 0.5)
        ctx.mm_set_accuracy(case["acc"])
        s["in"] = _bubble(case, seed)
    elif kind == "amr":
        nx, ny = case["nx"], case["ny"]
        cap = 8 * nx * ny
        ctx.mesh_rectangle(nx, ny, bounds=BOUNDS["periodic"])
        ctx.reserve(cap)
        ctx.configure(acc=2, flux="hllc", limiter=case["limiter"], cfl=0.5, gamma=GAMMA)
        ctx.set_state(*_carried(*_grid(nx, ny), seed))
        # a buffer for meshes up to the reserved size, read into after each cycle
        s["out"] = torch.zeros(5, cap, dtype=torch.float64, device="cuda")
        for _ in range(case["max_level"] + 2):   # the mesh of a running simulation
            _adapt_cycle(ctx, case)
    else:   # rect, adjoint
        ctx.mesh_rectangle(case["nx"], case["ny"], bounds=BOUNDS[case.get("bounds", "open")])
        ctx.configure(acc=case.get("acc", 2), flux=case.get("flux", "hllc"), limiter=case["limiter"], cfl=0.5,
                      gamma=GAMMA)
        st = _state2(case, seed)
        s["in"] = _on_gpu(st)
        s["out"] = torch.empty(5, ctx.n, dtype=torch.float64, device="cuda")
        if kind == "adjoint":
            s["window"] = (0.4, 0.6, 0.4, 0.6)
    return s


def _rows(t):
    n, p = t.shape[1], t.data_ptr()
    return [p + 8 * n * k for k in range(5)]


def _read(ctx, out):
    """The state into a device tensor of at least ctx.n columns."""
    if ctx.n > out.shape[1]:
        raise RuntimeError("the mesh outgrew the buffer")
    code = Z.lib().zfv_state_download_device(ctx.h, *[C.c_void_p(p) for p in _rows(out)])
    if code != Z.ZFV_OK:
        raise Z.ZfvError(code, Z.lib().zfv_last_error().decode())
    return out


def run(s):
    case, ctx = s["case"], s["ctx"]
    kind = case["kind"]
    if kind == "rect":
        ctx.set_state_device(_rows(s["in"]))
        ctx.step(case["steps"])
        return _read(ctx, s["out"]), ctx.dt()
    if kind == "batch":
        ctx.set_state_device(_rows(s["in"]))
        ctx.step(case["steps"])
        return _read(ctx, s["out"]), ctx.batch_dt()
    if kind == "adjoint":
        ctx.set_state_device(_rows(s["in"]))
        J = ctx.adjoint_forward(case["steps"], case["every"], s["window"])
        return [J] + ctx.adjoint_backward()
    if kind == "amr":
        _adapt_cycle(ctx, case)
        return _read(ctx, s["out"]), ctx.n
    if kind == "mm":
        ctx.mm_set_state(*s["in"])
        ctx.mm_step(case["steps"])
        return ctx.mm_state()
    ctx.step(case["steps"])
    return ctx.state()


# ---- what a pass cannot do without ----------------------------------------------
# Per cell and step: the state read once and written once, with the cell's
# volume and width; the operations of the scheme with every face evaluated once
# (a division or a square root counted as one).  Reading and setting a state
# moves it once each way.
def _cells(case):
    if case["kind"] == "batch":
        return sum(n * n for n in _sides(case))
    n = case["nx"] * case["ny"] * case.get("nz", 1)
    if case["kind"] == "amr":
        # the band of refined cells along the bubble's rim
        rim = 2.0 * math.pi * 0.2
        for level in range(1, case["max_level"] + 1):
            n += int(6.0 * rim * math.sqrt(case["nx"] * case["ny"]) * 2 ** level)
    return n


def work(case):
    kind, n, steps = case["kind"], _cells(case), case["steps"]
    if kind in ("rect", "batch"):
        flops = 2 * 80 + 60 if case.get("acc", 2) == 1 else 2 * 150 + 420
        return {"bytes": n * (steps * (2 * 44.0 + 16.0) + 2 * 80.0), "flops": float(n * steps * flops)}
    if kind == "adjoint":
        # forward, recompute and reverse, each reading and writing the state
        return {"bytes": n * steps * (3 * 104.0 + 80.0), "flops": float(n * steps * (2 * 720 + 3 * 720))}
    if kind == "amr":
        # the mesh of an adaptive step cannot come from tables: slots and centres too
        mesh = 4 + 16 + 4 * (4 + 3 * 8 + 8)
        return {"bytes": n * (steps * (104.0 + mesh) + 2 * (mesh + 2 * 9 * 8) + 80.0), "flops": float(n * steps * 720)}
    if kind == "mm":
        per = 2 * 8 * 11 + 16.0
        flops = 700 if case.get("acc", 1) == 1 else 2200
        return {"bytes": n * (steps * per + 15 * 8.0), "flops": float(n * steps * flops)}
    flops = 3 * 100 + 70 if case["acc"] == 1 else 3 * 210 + 700
    return {"bytes": n * (steps * (2 * 52.0 + 8.0) + 48.0), "flops": float(n * steps * flops)}


def tolerance(case):
    """Rounding at another place, carried through the steps of a pass: four
    times the largest difference from exact(), or (adaptive and two-material
    cases) between passes whose inputs differ by an ulp, over 60 drawn cases."""
    if case["kind"] == "adjoint":
        return {"rel": 1.5e-13, "max": 5e-12}
    if case["kind"] == "mm":
        return {"rel": 2e-12, "max": 2e-10}
    return {"rel": 3e-13, "max": 1e-12}


# ---- the same in plain torch ------------------------------------------------------
def _limit(name, a, b):
    """limiter(a, b) b of the reference's limiters."""
    if name == "minmod":
        return torch.where(a * b <= 0.0, 0.0 * b, torch.where(a.abs() < b.abs(), a, b))
    if name == "vanLeer":
        ok = (a * b > 0.0)
        den = torch.where(ok, a.abs() + b.abs(), torch.ones_like(a))
        return torch.where(ok, 2.0 * a.abs() / den * b, 0.0 * b)
    ok = (b != 0.0) & (a * b > 0.0)
    r = torch.where(ok, a, torch.zeros_like(a)) / torch.where(ok, b, torch.ones_like(b))
    two = torch.full_like(r, 2.0)
    mid = 0.5 * (1.0 + r) if name == "MC" else (1.0 + 2.0 * r) / 3.0
    return torch.where(ok, torch.minimum(2.0 * r, torch.minimum(mid, two)), torch.zeros_like(r)) * b


class _Exact:
    """MUSCL-Hancock (or first-order) step on a uniform grid of 2 or 3
    dimensions.  State z: (2 + d + 1, *shape) rows rho, velocities, p, e."""

    def __init__(self, shape, bounds, acc, flux, limiter, cfl=0.5):
        self.d, self.shape, self.bounds = len(shape), shape, bounds
        self.h = [1.0 / n for n in shape]
        self.acc, self.flux, self.limiter, self.cfl = acc, flux, limiter, cfl

    def edge(self, f, a, up, own):
        """f across the up (or down) side along axis a; `own` at a boundary."""
        n = f.shape[a + 1]
        g = torch.roll(f, -1 if up else 1, a + 1)
        if self.bounds[2 * a + (1 if up else 0)] == PERIODIC:
            return g
        at = torch.zeros(n, dtype=torch.bool, device=f.device)
        at[n - 1 if up else 0] = True
        at = at.reshape([1] + [n if k == a else 1 for k in range(self.d)])
        return torch.where(at, own, g)

    def mirror(self, z, a, up):
        if self.bounds[2 * a + (1 if up else 0)] != WALL:
            return z
        sign = torch.ones(z.shape[0], dtype=z.dtype, device=z.device)
        sign[1 + a] = -1.0
        return z * sign.reshape([-1] + [1] * self.d)

    def energy(self, z):
        e = z[self.d + 1] / ((GAMMA - 1.0) * z[0])
        return torch.cat([z[:self.d + 2], e[None]])

    def face_state(self, z, g, a, sgn):
        """z moved to the face centre by its gradient, or z itself where that
        is no state."""
        f = self.energy(z[:self.d + 2] + (0.5 * sgn * self.h[a]) * g[a])
        bad = (f[0] <= 0.0) | (f[self.d + 1] < 0.0)
        return torch.where(bad, z, f)

    def conserved(self, z):
        v = z[1:1 + self.d]
        return torch.cat([z[:1], z[0] * v, (z[0] * (z[self.d + 2] + 0.5 * (v * v).sum(0)))[None]])

    def primitive(self, q):
        v = q[1:1 + self.d] / q[0]
        e = q[self.d + 1] / q[0] - 0.5 * (v * v).sum(0)
        return torch.cat([q[:1], v, ((GAMMA - 1.0) * q[0] * e)[None], e[None]])

    def phys(self, z, a):
        q, vn, p = self.conserved(z), z[1 + a], z[self.d + 1]
        f = q * vn
        return torch.cat([f[:1 + a], (f[1 + a] + p)[None], f[2 + a:1 + self.d], (f[self.d + 1] + p * vn)[None]])

    def riemann(self, L, R, a):
        d = self.d
        p_L, p_R, u_L, u_R = L[d + 1], R[d + 1], L[1 + a], R[1 + a]
        c_L, c_R = torch.sqrt(GAMMA * p_L / L[0]), torch.sqrt(GAMMA * p_R / R[0])
        S_L, S_R = torch.minimum(u_L - c_L, u_R - c_R), torch.maximum(u_L + c_L, u_R + c_R)
        F_L, F_R, Q_L, Q_R = self.phys(L, a), self.phys(R, a), self.conserved(L), self.conserved(R)
        zero = torch.zeros_like(S_L)
        if self.flux == "rusanov":
            S = torch.maximum(torch.minimum(S_L, zero).abs(), torch.maximum(S_R, zero))
            return 0.5 * (F_L + F_R) + 0.5 * S * (Q_L - Q_R)
        if self.flux == "hll":
            S_L, S_R = torch.minimum(S_L, zero), torch.maximum(S_R, zero)
            return (S_R * F_L - S_L * F_R + S_L * S_R * (Q_R - Q_L)) / (S_R - S_L)
        a_L, a_R = L[0] * (S_L - u_L), R[0] * (S_R - u_R)
        S_C = (p_L - p_R + a_R * u_R - a_L * u_L) / (a_R - a_L)

        def star(z, q, A, S, u, p):
            r = A / (S - S_C)
            v = torch.cat([z[1:1 + a], S_C[None], z[2 + a:1 + d]])
            return torch.cat([r[None], r * v, (r * (q[d + 1] / z[0] + (S_C - u) * (S_C + p / A)))[None]])

        Qs_L, Qs_R = star(L, Q_L, a_L, S_L, u_L, p_L), star(R, Q_R, a_R, S_R, u_R, p_R)
        F = 0.5 * (F_L + F_R + S_L * (Qs_L - Q_L) + S_C.abs() * (Qs_L - Qs_R) + S_R * (Qs_R - Q_R))
        return torch.where(S_L >= 0.0, F_L, torch.where(S_R <= 0.0, F_R, F))

    def dt(self, z):
        v = z[1:1 + self.d]
        return self.cfl * (min(self.h) / (torch.sqrt((v * v).sum(0)) + torch.sqrt(GAMMA * z[self.d + 1] / z[0]))).min()

    def step(self, z):
        dt, d = self.dt(z), self.d
        if self.acc == 1:
            q = self.conserved(z)
            for a in range(d):
                for up in (False, True):
                    o = self.edge(z, a, up, self.mirror(z, a, up))
                    F = self.riemann(z, o, a) if up else -self.riemann(o, z, a)
                    q = q - dt / self.h[a] * F
            return self.primitive(q), dt
        w, g = z[:d + 2], []
        for a in range(d):
            h = self.h[a]
            up = self.edge(w, a, True, self.mirror(w, a, True)) - w
            dn = self.edge(w, a, False, self.mirror(w, a, False)) - w
            s = (up - dn) / (2.0 * h)
            g.append((_limit(self.limiter, 2.0 * s * h - up, up) - _limit(self.limiter, -2.0 * s * h - dn, dn)) /
                     (2.0 * h))
        q = self.conserved(z)
        for a in range(d):
            q = q - 0.5 * dt / self.h[a] * (self.phys(self.face_state(z, g, a, 1.0), a) -
                                            self.phys(self.face_state(z, g, a, -1.0), a))
        half = self.primitive(q)
        bad = (half[0] <= 0.0) | (half[d + 1] < 0.0)
        half = torch.where(bad, z, half)
        q = self.conserved(z)
        for a in range(d):
            hi, lo = self.face_state(half, g, a, 1.0), self.face_state(half, g, a, -1.0)
            over = self.edge(lo, a, True, self.mirror(hi, a, True))
            under = self.edge(hi, a, False, self.mirror(lo, a, False))
            q = q - dt / self.h[a] * (self.riemann(hi, over, a) - self.riemann(under, lo, a))
        return self.primitive(q), dt

    def steps(self, z, n):
        dt = None
        for _ in range(n):
            z, dt = self.step(z)
        return z, dt


def exact(case, seed):
    """The pass in plain torch.  None for the adaptive and the multi-material
    cases: their meshes and per-cell closures in plain torch take far longer
    than a pass may."""
    kind = case["kind"]
    if kind in ("amr", "mm"):
        return None
    if kind == "cube":
        shape = (case["nx"], case["ny"], case["nz"])
        E = _Exact(shape, BOUNDS3[case["bounds"]], case["acc"], case["flux"], case["limiter"])
        z, _ = E.steps(_on_gpu(_blast3(case, seed)).reshape(6, *shape), case["steps"])
        return list(z.reshape(6, -1))
    if kind == "batch":
        st, where = _batch_state(case, seed)
        out, dts = _on_gpu(st), []
        for n, b in where:
            E = _Exact((n, n), BOUNDS["open"], 2, "hllc", case["limiter"])
            z, dt = E.steps(out[:, b:b + n * n].reshape(5, n, n), case["steps"])
            out[:, b:b + n * n] = z.reshape(5, -1)
            dts.append(float(dt))
        return out, np.array(dts)
    shape = (case["nx"], case["ny"])
    z = _on_gpu(_state2(case, seed)).reshape(5, *shape)
    E = _Exact(shape, BOUNDS[case.get("bounds", "open")], case.get("acc", 2), case.get("flux", "hllc"),
               case["limiter"])
    if kind == "rect":
        z, dt = E.steps(z, case["steps"])
        return z.reshape(5, -1), float(dt)
    z = z.clone().requires_grad_(True)
    x, y = (torch.from_numpy(g.reshape(shape)).cuda() for g in _grid(*shape))
    inside = (x >= 0.4) & (x <= 0.6) & (y >= 0.4) & (y <= 0.6)
    f, _ = E.steps(z, case["steps"])
    J = (f[3] ** 2 * inside).sum() * (E.h[0] * E.h[1])
    (lam,) = torch.autograd.grad(J, z)
    return [float(J.detach())] + list(lam.reshape(5, -1))
