"""Performance cases: the work a user of fluam_amd has it do, through its public entry points.

A step case is one sampling interval of a run: a Simulation (or a Batch of them) whose state is
resident on the GPU takes `steps` time steps, is checked with sync(), and the sampled state is read
back the way an analysis program reads it.  The sampling intervals (50 and 100 steps) are the
`samplefreq` values of the data.main files under tests/golden.  A transform case is one call of the
forward FFT on caller-owned device buffers.

exact() restates the three schemes in 64-bit torch: the same Philox counter generator, Peskin
kernels, WCA force, staggered operators and Fourier-space solves.
"""
import ctypes as C
import math
import random

import numpy as np
import torch

import fluam_amd as F
from fluam_amd import (make_params, SCHEME_INCOMPRESSIBLE, SCHEME_QUASI_NEUTRALLY_BUOYANT, SCHEME_STOKES_LIMIT)

SCHEMES = {"incompressible": SCHEME_INCOMPRESSIBLE, "inertial": SCHEME_QUASI_NEUTRALLY_BUOYANT,
           "stokes": SCHEME_STOKES_LIMIT}
RC = 2.0 ** (1.0 / 6.0)  # WCA cutoff in units of sigma


def _sim(name, kind, cells, steps, np=0, kernel=3, h=1.0, kT=1e-3, dt=0.05, mass=0.0, mobility=0.0, graph=False,
         field=True, spectrum=False):
    """One simulation: h is the cell size, kernel the Peskin kernel's points, field whether the
    program samples the velocity field too, spectrum whether it samples S(k) every ten steps."""
    return dict(name=name, kind=kind, mx=cells[0], my=cells[1], mz=cells[2], steps=steps, np=np, kernel=kernel, h=h,
                kT=kT, dt=dt, mass=mass, mobility=mobility, graph=graph, field=field, spectrum=spectrum)


def listed():
    return [
        # one forward transform on device buffers, as code that cannot allocate calls it
        dict(name="transform_96", kind="transform", mx=96, my=96, mz=96),
        # fluam's example inputs: a 32^3 box at equilibrium, and the same box with one heavy particle
        _sim("incompressible_32", "incompressible", (32, 32, 32), 50, h=10.0, kT=0.1, dt=0.25),
        _sim("inertial_32_one", "inertial", (32, 32, 32), 50, np=1, h=10.0, kT=0.1, dt=0.25, mass=8000.0),
        # a small suspension run for long times: graph replay
        _sim("stokes_32_graph", "stokes", (32, 32, 32), 100, np=1024, graph=True),
        # the inertial-coupling configuration: particles and flow sampled
        _sim("inertial_64", "inertial", (64, 64, 64), 100, np=4096),
        # a dense suspension, flow sampled
        _sim("stokes_64_dense", "stokes", (64, 64, 64), 100, np=16384, kernel=4),
        # a ragged box of the fluid alone, its structure factor accumulated in place
        _sim("incompressible_ragged", "incompressible", (108, 54, 72), 50, spectrum=True),
        # particles denser than the fluid in a rectangular box
        _sim("inertial_heavy_rect", "inertial", (96, 48, 64), 50, np=6000, kernel=4, mass=2.0),
        # a thin slab with extra particle mobility
        _sim("stokes_slab", "stokes", (128, 64, 32), 100, np=8192, mobility=0.05),
        # an ensemble of small unequal boxes stepped together
        dict(name="batch_32", kind="batch", replicas=32, mix=4, steps=50, kernel=3, kT=1e-3, dt=0.05, h=1.0),
        # the headline configuration: particle trajectories
        _sim("stokes_128", "stokes", (128, 128, 128), 100, np=65536, kernel=4, field=False),
        # the largest box
        _sim("stokes_largest", "stokes", (128, 128, 256), 100, np=131072, kernel=4, field=False),
    ]


def draw(rng):
    kind = rng.choice(("incompressible", "inertial", "stokes", "inertial", "stokes", "stokes", "batch", "transform"))
    if kind == "batch":
        return dict(kind="batch", replicas=rng.randint(4, 32), mix=rng.randrange(1 << 20), steps=50,
                    kernel=rng.choice((3, 4)), kT=1e-3, dt=0.05, h=1.0)
    even = (16, 24, 32, 36, 48, 64, 72, 96, 108, 128)
    odd = (18, 27, 54, 81)
    while True:
        free = even + odd if kind in ("incompressible", "transform") else even
        if rng.random() < 0.4:  # cubes are the usual choice
            mx = my = mz = rng.choice(even)
        else:
            mx = rng.choice([m for m in free if m % 2 == 0])
            my, mz = rng.choice(free), rng.choice(free + (144, 192, 256))
        if (mx // 2 + 1) * my > 8448 or mx * my * mz > 128 ** 3:
            continue
        if kind == "transform":
            if mz * my * (mx // 2 + 1) > 128 * 128 * 65:
                continue
            return dict(kind="transform", mx=mx, my=my, mz=mz)
        N = mx * my * mz
        if kind == "incompressible":
            c = _sim("", kind, (mx, my, mz), rng.choice((50, 100)), spectrum=rng.random() < 0.3)
        else:
            top = min(N // 16, 65536)
            n = int(round(math.exp(rng.uniform(0.0, math.log(top)))))
            heavy = kind == "inertial" and rng.random() < 0.3
            if heavy and N > 64 * 64 * 128:
                continue
            c = _sim("", kind, (mx, my, mz), rng.choice((50, 100)), np=n, kernel=rng.choice((3, 4)),
                     mass=2.0 if heavy else 0.0, mobility=0.05 if kind == "stokes" and rng.random() < 0.3 else 0.0,
                     field=kind == "inertial" or rng.random() < 0.3)
        c["graph"] = rng.random() < 0.25
        del c["name"]
        return c


# ---------------------------------------------------------------------------------------
# What the program has in hand: parameters, start state, contexts.
# ---------------------------------------------------------------------------------------
def _params(c, seed):
    sigma = 1.0 if c["h"] == 1.0 else 2.0 * c["h"]
    cells = (c["mx"], c["my"], c["mz"])
    kw = dict(temperature=c["kT"], dt=c["dt"], seed=1 + seed)
    if c["np"]:
        kw.update(np=c["np"], kernel_points=c["kernel"], initial_positions=1, cutoff=RC * sigma, wca_sigma=sigma,
                  mass=c["mass"], extra_mobility=c["mobility"])
    return make_params(SCHEMES[c["kind"]], cells=cells, box=tuple(c["h"] * m for m in cells), **kw)


def _start(p, seed):
    """Start positions (np, 3) and velocity (3, mz, my, mx) of a run: particles on randomly chosen
    sites of a lattice of 1.25 sigma, displaced by up to 0.12 sigma (no pair starts inside the WCA
    core, some start within its range); the fluid at thermal equilibrium."""
    rng = np.random.default_rng((seed, p.mx, p.my, p.mz, p.np))
    box = np.array((p.lx, p.ly, p.lz))
    q = None
    if p.np:
        a = 1.25 * p.wca_sigma
        sites = np.maximum((box / a).astype(int), 1)
        pick = rng.choice(int(sites.prod()), p.np, replace=False)
        at = np.stack(np.unravel_index(pick, sites), 1)
        q = (at + 0.5) * (box / sites) - 0.5 * box + rng.uniform(-0.12, 0.12, (p.np, 3)) * p.wca_sigma
    v = None
    if p.scheme != SCHEME_STOKES_LIMIT:
        dV = (p.lx / p.mx) * (p.ly / p.my) * (p.lz / p.mz)
        v = rng.standard_normal((3, p.mz, p.my, p.mx), dtype=np.float32)
        v *= np.float32(math.sqrt(p.temperature / (p.densfluid * dV)))
        v -= v.mean(axis=(1, 2, 3), keepdims=True)
    return q, v


def _members(c):
    """The simulations of a batch: Stokes-limit boxes with edges drawn per axis from the ensemble's
    lengths and up to 2048 particles."""
    rng = random.Random(c["mix"])
    out = []
    for _ in range(c["replicas"]):
        cells = tuple(rng.choice((16, 24, 32, 48, 64)) for _ in range(3))
        n = rng.randint(1, min(2048, cells[0] * cells[1] * cells[2] // 8))
        out.append(_sim("", "stokes", cells, c["steps"], np=n, kernel=c["kernel"], h=c["h"], kT=c["kT"], dt=c["dt"]))
    return out


def _transform_input(c, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    return torch.randn((c["mz"], c["my"], c["mx"]), generator=g, device="cuda")


def prepare(case, seed):
    c = case
    if c["kind"] == "transform":
        fft = F.lib().fhd_fft_r2c_noalloc
        fft.argtypes = [C.c_int, C.c_int, C.c_int, C.c_void_p, C.c_void_p, C.c_void_p]
        x = _transform_input(c, seed)
        out = torch.empty((c["mz"], c["my"], c["mx"] // 2 + 1), dtype=torch.complex64, device="cuda")
        return {"case": c, "fft": fft, "x": x, "out": out}
    if c["kind"] == "batch":
        ps = [_params(m, 64 * seed + i) for i, m in enumerate(_members(c))]
        b = F.Batch(ps)
        b.set_mode(2)
        for i, (p, s) in enumerate(zip(ps, b.replicas)):
            s.set_particles(_start(p, 64 * seed + i)[0].T.ravel())
        return {"case": c, "batch": b, "close": _Closer(b)}
    p = _params(c, seed)
    sim = F.Simulation(p)
    q, v = _start(p, seed)
    if v is not None:
        sim.set_velocity(v.ravel())
    if q is not None:
        sim.set_particles(q.T.ravel())
    if c["graph"]:
        sim.set_graph(True)
    return {"case": c, "sim": sim}


class _Closer:
    """Gives a batch's memory back when its state is dropped."""

    def __init__(self, b):
        self.b = b

    def __del__(self):
        self.b.close()


def run(state):
    c = state["case"]
    if c["kind"] == "transform":
        stream = torch.cuda.current_stream().cuda_stream
        ok = state["fft"](c["mx"], c["my"], c["mz"], state["x"].data_ptr(), state["out"].data_ptr(), stream)
        if not ok:
            raise RuntimeError(F.lib().fhd_last_error().decode())
        return state["out"]
    f32 = np.float32  # the fields are 32-bit on the device
    if c["kind"] == "batch":
        b = state["batch"]
        b.step(c["steps"])
        b.sync()
        return {"positions": np.concatenate([s.particles() for s in b.replicas]).astype(f32),
                "velocities": np.concatenate([s.particle_velocities() for s in b.replicas]).astype(f32)}
    sim = state["sim"]
    if c["spectrum"]:
        sim.sk_reset()
        for _ in range(c["steps"] // 10):
            sim.step(10)
            sim.sk_sample()
    else:
        sim.step(c["steps"])
    sim.sync()
    out = {}
    if c["spectrum"]:
        out["spectrum"] = sim.structure_factor()[0].astype(f32)
    if c["field"]:
        out["velocity"] = sim.velocity().astype(f32)
    if c["np"]:
        out["positions"] = sim.particles().astype(f32)
        out["velocities"] = sim.particle_velocities().astype(f32)
        out["forces"] = sim.forces().astype(f32)
    return out


def work(case):
    """Per step, the fields that have to pass between the dependent stages (FP32, three components,
    the noise generated in place): a spread or right-hand side written into the xy transform, the
    half spectrum written, read and written by the solve and read by the inverse, the velocity
    written, and read by the stages that use it."""
    c = case
    if c["kind"] == "transform":
        N, half = c["mx"] * c["my"] * c["mz"], c["my"] * c["mz"] * (c["mx"] // 2 + 1)
        return {"bytes": 4 * N + 8 * half, "flops": 2.5 * N * math.log2(N)}
    if c["kind"] == "batch":
        ws = [work(m) for m in _members(c)]
        return {"bytes": sum(w["bytes"] for w in ws), "flops": sum(w["flops"] for w in ws)}
    N, n = c["mx"] * c["my"] * c["mz"], c["np"]
    heavy = c["mass"] != 0.0
    cell, part, solves = {"incompressible": (168, 0, 2), "stokes": (192, 200, 2),
                          "inertial": (132 + (270 if heavy else 0), 200 + (400 if heavy else 0), 3 if heavy else 1)}[c["kind"]]
    per_node = 3 * c["kernel"] ** 3
    b = c["steps"] * (cell * N + part * n)
    f = c["steps"] * (solves * (6 * 2.5 * N * math.log2(N) + 60 * N) + 2 * solves * 2 * per_node * n)
    return {"bytes": b, "flops": f}


# ---------------------------------------------------------------------------------------
# The same steps in 64-bit torch.
# ---------------------------------------------------------------------------------------
M32 = 0xFFFFFFFF


def _philox(c0, c1, step, seed):
    """Philox4x32-10 of counters (c0, c1, step low, step high), key = seed."""
    x, y = c0, torch.full_like(c0, c1)
    z, w = torch.full_like(c0, step & M32), torch.full_like(c0, (step >> 32) & M32)
    k0, k1 = seed & M32, (seed >> 32) & M32
    for _ in range(10):
        p0, p1 = x * 0xD2511F53, z * 0xCD9E8D57
        x, y, z, w = ((p1 >> 32) & M32) ^ y ^ k0, p1 & M32, ((p0 >> 32) & M32) ^ w ^ k1, p0 & M32
        k0, k1 = (k0 + 0x9E3779B9) & M32, (k1 + 0xBB67AE85) & M32
    return x, y, z, w


def _normals4(index, stream, sub, step, seed):
    w = _philox(index, (stream << 4) | sub, step, seed)
    out = []
    for a, b in ((w[0], w[1]), (w[2], w[3])):
        r = torch.sqrt(-2.0 * torch.log(((a >> 8) + 1).double() / 2 ** 24))
        t = 2.0 * math.pi * (b >> 8).double() / 2 ** 24
        out += [r * torch.cos(t), r * torch.sin(t)]
    return out


def _phi(r, pts):
    r = r.abs()
    if pts == 3:
        near = (1 + torch.sqrt((1 - 3 * r * r).clamp(min=0))) / 3
        far = (5 - 3 * r - torch.sqrt((1 - 3 * (1 - r) ** 2).clamp(min=0))) / 6
        return torch.where(r < 0.5, near, torch.where(r < 1.5, far, 0 * r))
    near = (3 - 2 * r + torch.sqrt((1 + 4 * r - 4 * r * r).clamp(min=0))) / 8
    far = (5 - 2 * r - torch.sqrt((-7 + 12 * r - 4 * r * r).clamp(min=0))) / 8
    return torch.where(r <= 1, near, torch.where(r < 2, far, 0 * r))


def _dphi(r, pts):
    s, r = torch.sign(r), r.abs()
    if pts == 3:
        near = -r / torch.sqrt((1 - 3 * r * r).clamp(min=1e-30))
        far = -0.5 * (1 + (1 - r) / torch.sqrt((-2 + 6 * r - 3 * r * r).clamp(min=1e-30)))
        return s * torch.where(r <= 0.5, near, torch.where(r < 1.5, far, 0 * r))
    near = (-2 + (2 - 4 * r) / torch.sqrt((1 + 4 * r - 4 * r * r).clamp(min=1e-30))) / 8
    far = (-2 - (6 - 4 * r) / torch.sqrt((-7 + 12 * r - 4 * r * r).clamp(min=1e-30))) / 8
    return s * torch.where(r <= 1, near, torch.where(r < 2, far, 0 * r))


class _Reference:
    """One run; fields (3, mz, my, mx), particles (np, 3), axis order x, y, z in component indices."""

    def __init__(self, p, q, v):
        self.p, self.dev = p, torch.device("cuda")
        self.m = (p.mx, p.my, p.mz)
        self.L = (p.lx, p.ly, p.lz)
        self.h = tuple(l / m for l, m in zip(self.L, self.m))
        self.dV = self.h[0] * self.h[1] * self.h[2]
        self.step_no = 0
        self.q = None if q is None else self.t(q)
        self.u = None if q is None else 0 * self.q
        self.F = self.u
        self.lag = self.u
        self.v = None if v is None else self.t(v)
        self.adv = None
        P = p.mx // 2 + 1
        g, e = [], []
        for a, n in enumerate((P, p.my, p.mz)):
            k = torch.arange(n, device=self.dev, dtype=torch.float64)
            shape = [1, 1, 1]
            shape[2 - a] = n
            g.append((2 / self.h[a] * torch.sin(math.pi * k / self.m[a])).reshape(shape))
            e.append(torch.exp(1j * math.pi * k / self.m[a]).reshape(shape))
        self.g, self.e = g, e
        self.g2 = g[0] ** 2 + g[1] ** 2 + g[2] ** 2
        if self.v is not None:
            self.v = self.solve(self.v, 0.0)

    def t(self, x):
        return torch.as_tensor(np.asarray(x), device=self.dev).double()

    # ---- fluid ----
    def solve(self, w, cn=None, noise=None):
        """cn: Crank-Nicolson coefficient (0: projection); None: the Stokes operator."""
        wh = list(torch.fft.rfftn(w, dim=(1, 2, 3)))
        if noise is not None:
            wh = [a + b for a, b in zip(wh, noise)]
        wh = [a * e.conj() for a, e in zip(wh, self.e)]
        g2 = self.g2.clone()
        g2[0, 0, 0] = 1.0
        gw = (self.g[0] * wh[0] + self.g[1] * wh[1] + self.g[2] * wh[2]) / g2
        gw[0, 0, 0] = 0
        if cn is None:
            den = 1 / (self.p.shearviscosity * g2)
            den[0, 0, 0] = 0
        else:
            den = 1 / (1 + cn * self.g2)
        out = torch.stack([(a - g * gw) * den * e for a, g, e in zip(wh, self.g, self.e)])
        return torch.fft.irfftn(out, s=(self.p.mz, self.p.my, self.p.mx), dim=(1, 2, 3))

    def sh(self, f, dx=0, dy=0, dz=0):
        """f at (x + dx, y + dy, z + dz)."""
        return torch.roll(f, (-dz, -dy, -dx), (-3, -2, -1))

    def laplacian(self, f):
        out = 0
        for a, d in enumerate(((1, 0, 0), (0, 1, 0), (0, 0, 1))):
            out = out + (self.sh(f, *d) - 2 * f + self.sh(f, *(-i for i in d))) / self.h[a] ** 2
        return out

    def advection(self, v):
        """(1/4) sum_b D_b[(v_a + v_a')(v_b + v_b')]: component a at its face."""
        unit = ((1, 0, 0), (0, 1, 0), (0, 0, 1))
        out = []
        for a in range(3):
            s = 0
            for b in range(3):
                up, dn = unit[b], tuple(-i for i in unit[b])
                va, vb = v[a], v[b]
                flux_up = (self.sh(va, *up) + va) * (self.sh(vb, *unit[a]) + vb)
                lo = tuple(i + j for i, j in zip(dn, unit[a]))
                flux_dn = (va + self.sh(va, *dn)) * (self.sh(vb, *lo) + self.sh(vb, *dn))
                if a == b:
                    flux_up = (self.sh(va, *up) + va) ** 2
                    flux_dn = (va + self.sh(va, *dn)) ** 2
                s = s + (flux_up - flux_dn) / self.h[b]
            out.append(0.25 * s)
        return torch.stack(out)

    def stress_divergence(self, f1, f4):
        p = self.p
        i = torch.arange(p.mx * p.my * p.mz, device=self.dev)
        n = [x.reshape(p.mz, p.my, p.mx) for k in (0, 1) for x in _normals4(i, 1, k, self.step_no, p.seed)]
        xx, xy, xz, yy, yz, zz = n[:6]
        tr = (xx + yy + zz) / 3
        xx, yy, zz = xx - tr, yy - tr, zz - tr
        hx, hy, hz = self.h
        s = self.sh
        return torch.stack([
            f1 / hx * (s(xx, 1) - xx) + f4 / hy * (xy - s(xy, 0, -1)) + f4 / hz * (xz - s(xz, 0, 0, -1)),
            f1 / hy * (s(yy, 0, 1) - yy) + f4 / hx * (xy - s(xy, -1)) + f4 / hz * (yz - s(yz, 0, 0, -1)),
            f1 / hz * (s(zz, 0, 0, 1) - zz) + f4 / hx * (xz - s(xz, -1)) + f4 / hy * (yz - s(yz, 0, -1))])

    def mode_noise(self, nset, f4):
        """The part of the Stokes step's noise that the solve keeps, per mode of the half spectrum."""
        p = self.p
        mx, my, mz = self.m
        P = mx // 2 + 1
        kz, ky, kx = torch.meshgrid(*(torch.arange(n, device=self.dev) for n in (mz, my, P)), indexing="ij")
        py, pz = (my - ky) % my, (mz - kz) % mz
        edge = (kx == 0) | (2 * kx == mx)
        a, b = ky + my * kz, py + my * pz
        selfc, conj = edge & (a == b), edge & (b < a)
        cy, cz = torch.where(conj, py, ky), torch.where(conj, pz, kz)
        g = [x.expand(mz, my, P) for x in self.g]
        e = [x.expand(mz, my, P) for x in self.e]
        e[1] = torch.where(conj & (ky != 0), -e[1].conj(), e[1])
        e[2] = torch.where(conj & (kz != 0), -e[2].conj(), e[2])
        on = [kx != 0, ky != 0, kz != 0]
        count = on[0].long() + on[1].long() + on[2].long()
        gn = torch.sqrt(self.g2)
        ig = 1 / gn.clamp(min=1e-300)
        t1, t2 = torch.zeros((3, mz, my, P), device=self.dev, dtype=torch.float64), None
        t2 = t1.clone()
        r = 1 / torch.sqrt((g[0] ** 2 + g[1] ** 2).clamp(min=1e-300))
        full = count == 3
        c1 = torch.stack([g[1] * r, -g[0] * r, 0 * r])
        c2 = torch.stack([-g[2] * c1[1], g[2] * c1[0], g[0] * c1[1] - g[1] * c1[0]]) * ig
        t1, t2 = torch.where(full, c1, t1), torch.where(full, c2, t2)
        im1, im2 = full.clone(), full.clone()
        for c in range(3):
            a, b = [i for i in range(3) if i != c]
            two = (count == 2) & ~on[c]
            t1[c] = torch.where(two, torch.ones_like(gn), t1[c])
            t2[a] = torch.where(two, -g[b] * ig, t2[a])
            t2[b] = torch.where(two, g[a] * ig, t2[b])
            im2 = im2 | two
            one = (count == 1) & on[c]
            t1[a] = torch.where(one, torch.ones_like(gn), t1[a])
            t2[b] = torch.where(one, torch.ones_like(gn), t2[b])
        index = (kx + P * (cy + my * cz)).reshape(-1)
        n = 0
        for s in range(nset):
            n = n + torch.stack(_normals4(index, 6, s, self.step_no, p.seed))
        n = n.reshape(4, mz, my, P)
        half = math.sqrt(0.5 * mx * my * mz)
        z1, z2 = half * torch.complex(n[0], n[1]), half * torch.complex(n[2], n[3])
        root2 = math.sqrt(2.0) * half
        i1, i2 = torch.where(im1, 1j, 1 + 0j), torch.where(im2, 1j, 1 + 0j)
        z1, z2 = torch.where(selfc, root2 * n[0] * i1, z1), torch.where(selfc, root2 * n[2] * i2, z2)
        w = []
        for k in range(3):
            x = f4 * gn * (z1 * t1[k] + z2 * t2[k]) * e[k]
            w.append(torch.where(count == 0, 0 * x, torch.where(conj, x.conj(), x)))
        return w

    # ---- particles ----
    def weights(self, q, deriv=False):
        """Per axis, node indices and weights at the centred and the face nodes."""
        pts = self.p.kernel_points
        k = torch.arange(pts, device=self.dev)
        out = []
        for a in range(3):
            pair = []
            for stag in (0, 1):
                u = (q[:, a] + 0.5 * self.L[a]) / self.h[a] - (1.0 if stag else 0.5)
                base = (torch.floor(u + 0.5) if pts == 3 else torch.floor(u)).long() - 1
                r = u[:, None] - (base[:, None] + k)
                w = _dphi(r, pts) if deriv and stag else _phi(r, pts)
                pair.append(((base[:, None] + k) % self.m[a], w))
            out.append(pair)
        return out

    def nodes(self, w, comp):
        (ix, wx), (iy, wy), (iz, wz) = (w[a][1 if a == comp else 0] for a in range(3))
        at = (iz[:, :, None, None] * self.m[1] + iy[:, None, :, None]) * self.m[0] + ix[:, None, None, :]
        return at.reshape(len(ix), -1), (wz[:, :, None, None] * wy[:, None, :, None] * wx[:, None, None, :]).reshape(len(ix), -1)

    def spread(self, q, val, deriv=False):
        w = self.weights(q, deriv)
        out = torch.zeros((3, self.m[0] * self.m[1] * self.m[2]), device=self.dev, dtype=torch.float64)
        for a in range(3):
            at, x = self.nodes(w, a)
            out[a].index_add_(0, at.reshape(-1), (x * val[:, a:a + 1]).reshape(-1))
        return out.reshape(3, self.m[2], self.m[1], self.m[0]) / self.dV

    def interp(self, q, f):
        w = self.weights(q)
        out = []
        for a in range(3):
            at, x = self.nodes(w, a)
            out.append((f[a].reshape(-1)[at] * x).sum(1))
        return torch.stack(out, 1)

    def wca(self, q):
        p, L = self.p, torch.tensor(self.L, device=self.dev, dtype=torch.float64)
        rc, n = p.cutoff, len(q)
        bins = [max(1, int(l / rc)) for l in self.L]
        assert min(bins) >= 3
        nb = torch.tensor(bins, device=self.dev)
        w = q / L + 0.5
        c = ((w - torch.floor(w)) * nb).long() % nb
        at = (c[:, 2] * bins[1] + c[:, 1]) * bins[0] + c[:, 0]
        order = torch.argsort(at)
        cnt = torch.bincount(at, minlength=bins[0] * bins[1] * bins[2])
        first = torch.cumsum(cnt, 0) - cnt
        most = int(cnt.max())
        table = torch.full((len(cnt), most), -1, device=self.dev)
        table[at[order], torch.arange(n, device=self.dev) - first[at[order]]] = order
        out = torch.zeros_like(q)
        i = torch.arange(n, device=self.dev)[:, None]
        for dz in (-1, 0, 1):
            for dy in (-1, 0, 1):
                for dx in (-1, 0, 1):
                    d = (c + torch.tensor([dx, dy, dz], device=self.dev)) % nb
                    j = table[(d[:, 2] * bins[1] + d[:, 1]) * bins[0] + d[:, 0]]
                    r = q[:, None, :] - q[j.clamp(min=0)]
                    r = r - L * torch.round(r / L)
                    r2 = (r * r).sum(2)
                    ok = (j >= 0) & (j != i) & (r2 < rc * rc) & (r2 > 0)
                    r2 = r2.clamp(min=1e-4 * p.wca_sigma ** 2)
                    s6 = (p.wca_sigma ** 2 / r2) ** 3
                    f = torch.where(ok, 48 * p.wca_epsilon * (s6 * s6 - 0.5 * s6) / r2, torch.zeros_like(r2))
                    out += (f[:, :, None] * r).sum(1)
        return out

    # ---- the schemes ----
    def noise_factors(self):
        p = self.p
        s = p.temperature * p.shearviscosity * p.dt / (self.dV * p.densfluid ** 2)
        return math.sqrt(4 * s), math.sqrt(2 * s), 0.5 * p.dt * p.shearviscosity / p.densfluid

    def incompressible(self):
        f1, f4, cn = self.noise_factors()
        w0 = self.v + cn * self.laplacian(self.v) + self.stress_divergence(f1, f4)
        star = 0.5 * (self.solve(w0 - self.p.dt * self.advection(self.v), cn) + self.v)
        self.v = self.solve(w0 - self.p.dt * self.advection(star), cn)

    def stokes(self):
        p = self.p
        f4 = math.sqrt(2 * p.temperature * p.shearviscosity / (self.dV * p.dt))
        ids = torch.arange(len(self.q), device=self.dev)
        q0, f0 = self.q, self.wca(self.q)
        v = self.solve(self.spread(q0, f0), None, self.mode_noise(1, math.sqrt(2) * f4))
        qh = q0 + 0.5 * p.dt * self.interp(q0, v)
        if p.extra_mobility:
            z1 = torch.stack(_normals4(ids, 4, 0, self.step_no, p.seed)[:3], 1)
            z2 = torch.stack(_normals4(ids, 5, 0, self.step_no, p.seed)[:3], 1)
            amp = math.sqrt(p.temperature * p.extra_mobility * p.dt)
            qh = qh + 0.5 * p.dt * p.extra_mobility * f0 + amp * z1
        self.F = self.wca(qh)
        n = torch.stack(_normals4(ids, 3, 0, self.step_no, p.seed)[:3], 1)
        k, d = p.temperature / p.rfd_delta, 0.5 * p.rfd_delta
        w = self.spread(qh, self.F) + self.spread(q0 + d * n, k * n) - self.spread(q0 - d * n, k * n)
        v = self.solve(w, None, self.mode_noise(2, math.sqrt(0.5) * f4))
        self.u = self.interp(qh, v)
        self.q = q0 + p.dt * self.u
        if p.extra_mobility:
            self.q = self.q + p.dt * p.extra_mobility * self.F + amp * (z1 + z2)
        self.v = v

    def heavy(self, qh, vt, lag):
        """Excess-mass corrections: (new particle velocity, dv)."""
        p = self.p
        du = (self.lag if lag else 0) + self.interp(qh, self.v) - self.interp(self.q, self.v)
        jvt = self.interp(qh, vt)
        dp = p.mass * (self.u - jvt - du)
        f = 1.5 * p.volume_particle / (1.5 * p.volume_particle * self.dV * p.densfluid + p.mass)
        jd = self.interp(qh, self.solve(self.spread(qh, f * self.dV * dp), 0.0))
        cn = 0.5 * p.dt * p.shearviscosity / p.densfluid
        dv = self.solve(self.spread(qh, (dp - p.mass * jd) / p.densfluid), cn)
        return jvt + jd + du, dv, cn * self.laplacian(dv)

    def inertial(self):
        p = self.p
        f1, f4, cn = self.noise_factors()
        qh = self.q + 0.5 * p.dt * self.interp(self.q, self.v)
        self.F = self.wca(qh)
        mf = 1.5 * self.dV * p.volume_particle * p.densfluid
        drift = p.temperature * mf / (p.mass + mf)
        inv_h = torch.tensor([1 / h for h in self.h], device=self.dev, dtype=torch.float64)
        sf = self.spread(qh, self.F) + self.spread(qh, (drift * inv_h).expand(len(qh), 3), deriv=True)
        w0 = self.v + cn * self.laplacian(self.v) + self.stress_divergence(f1, f4) + p.dt / p.densfluid * sf
        adv = self.advection(self.v)
        if self.adv is None:
            vt = self.solve(w0 - p.dt * adv, cn)
            half = 0.5 * (self.v + vt)
            if p.mass:
                _, dv, lap = self.heavy(qh, vt, False)
                half = half + 0.5 * dv
                self.lag = self.interp(self.q + 0.5 * p.dt * self.interp(qh, half), lap)
            w = w0 - p.dt * self.advection(half)
        else:
            w = w0 - 1.5 * p.dt * adv + 0.5 * p.dt * self.adv
        self.adv = adv
        v2 = self.solve(w, cn)
        if p.mass:
            self.u, dv, lap = self.heavy(qh, v2, True)
            v2 = v2 + dv
            self.lag = self.interp(qh, lap)
        else:
            self.u = self.interp(qh, v2)
        self.q = self.q + 0.5 * p.dt * (self.interp(qh, self.v) + self.interp(qh, v2))
        self.v = v2

    def advance(self, steps):
        f = {SCHEME_INCOMPRESSIBLE: self.incompressible, SCHEME_QUASI_NEUTRALLY_BUOYANT: self.inertial,
             SCHEME_STOKES_LIMIT: self.stokes}[self.p.scheme]
        for _ in range(steps):
            f()
            self.step_no += 1

    def spectrum(self):
        s = torch.fft.rfftn(self.v, dim=(1, 2, 3))
        return (s.real ** 2 + s.imag ** 2) * self.p.densfluid * self.dV / (self.p.temperature * self.v[0].numel())


def _host(x):
    return x.cpu().numpy()


def exact(case, seed):
    c = case
    if c["kind"] == "transform":
        return torch.fft.rfftn(_transform_input(c, seed).double(), dim=(0, 1, 2))
    if c["kind"] == "batch":
        q, u = [], []
        for i, m in enumerate(_members(c)):
            p = _params(m, 64 * seed + i)
            r = _Reference(p, *_start(p, 64 * seed + i))
            r.advance(c["steps"])
            q.append(r.q.T.reshape(-1))
            u.append(r.u.T.reshape(-1))
        return {"positions": _host(torch.cat(q)), "velocities": _host(torch.cat(u))}
    p = _params(c, seed)
    r = _Reference(p, *_start(p, seed))
    out, s = {}, 0
    if c["spectrum"]:
        for _ in range(c["steps"] // 10):
            r.advance(10)
            s = s + r.spectrum()
        out["spectrum"] = _host(s / (c["steps"] // 10))
    else:
        r.advance(c["steps"])
    if c["field"]:
        out["velocity"] = _host(r.v.reshape(-1))
    if c["np"]:
        out["positions"] = _host(r.q.T.reshape(-1))
        out["velocities"] = _host(r.u.T.reshape(-1))
        out["forces"] = _host(r.F.T.reshape(-1))
    return out
