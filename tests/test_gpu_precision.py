"""Rounding errors of whole runs against the FP64 oracle.

The fluid's velocity is kept in 32 bits: 50 steps that each round it to 2.4e-8 of itself leave 1.7e-7,
the steps' changes (a fifth of the velocity, through transforms good to 2e-7) 2.8e-7 and the noise's own
6e-8: 3.4e-7 together.  Bound: three times that, 1e-6, for the field and for the root mean square over
seeds of a particle's three numbers.  The kept part of the velocity is projected again step by step, so its
divergence stays at the rounding error of the velocity, 6e-8 sqrt(6) / h of it, times 1 / sqrt(1 - s^2) =
5.7 for a kept share s of 63/64: 8.4e-7 root mean square over the cells, and five times that at the worst of
4096 of them."""
import numpy as np
import pytest

import fluam_amd as F
import oracle_lib as O
from fluam_amd._abi import (make_params, SCHEME_INCOMPRESSIBLE, SCHEME_QUASI_NEUTRALLY_BUOYANT,
                            SCHEME_STOKES_LIMIT)

pytestmark = pytest.mark.gpu


def rel(a, b):
    return np.linalg.norm(a - b) / np.linalg.norm(b)


def pair(scheme, cells, seed, h, kT, dt, **kw):
    """Both sides of a run that starts at thermal equilibrium."""
    print(f"[gpu-case] precision scheme={scheme} cells={cells} seed={seed}", flush=True)
    p = make_params(scheme, cells=cells, box=tuple(h * m for m in cells), temperature=kT, dt=dt, seed=seed, **kw)
    rng = np.random.default_rng(seed)
    v = rng.standard_normal(3 * cells[0] * cells[1] * cells[2]) * np.sqrt(kT / h ** 3)
    v = v.astype(np.float32).astype(np.float64)
    g, o = F.Simulation(p), O.Oracle(p)
    g.set_velocity(v)
    o.set_velocity(v)
    return p, rng, g, o


@pytest.mark.parametrize("mx", [16, 48, 54, 96, 128, 256])
def test_forward_transform_of_a_point_gives_the_nearest_twiddles(mx):
    """A point next to the origin transforms to e^{-2 pi i k / mx}: 32-bit twiddles rounded to nearest are off
    by at most 2^-25 a component, 2^-25 / sqrt(3) root mean square, and nothing else rounds on the way."""
    a = np.zeros((16, 16, mx))
    a[0, 0, 1] = 1.0
    off = F.fft_r2c(a)[0, 0] - np.exp(-2j * np.pi * np.arange(mx // 2 + 1) / mx)
    assert max(abs(off.real).max(), abs(off.imag).max()) < 1.0001 * 2.0 ** -25
    assert np.sqrt(np.mean(np.abs(off) ** 2)) < np.sqrt(2.0 / 3.0) * 2.0 ** -25


def test_particle_velocity_of_a_heavy_particle():
    off = []
    for seed in range(6):
        p, rng, g, o = pair(SCHEME_QUASI_NEUTRALLY_BUOYANT, (32, 32, 32), 3 + seed, 10.0, 0.1, 0.25, np=1,
                            kernel_points=3, mass=8000.0, initial_positions=1, nonbonded=0, cutoff=0.0)
        q = rng.uniform(-150.0, 150.0, 3)
        g.set_particles(q)
        o.set_particles(q)
        g.step(50)
        g.sync()
        o.step(50)
        off.append(rel(g.particle_velocities(), o.particle_velocities()))
        assert rel(g.velocity(), o.velocity()) < 1e-6
    print("  u", " ".join("%.1e" % x for x in off), flush=True)
    assert np.sqrt(np.mean(np.square(off))) < 1e-6


@pytest.mark.parametrize("cells,h,dt,plan", [
    ((32, 32, 32), 10.0, 0.25, None),
    ((48, 24, 16), 1.0, 0.05, None),
    ((96, 96, 8), 10.0, 0.25, None),
    ((128, 128, 4), 10.0, 0.25, None),
    ((128, 128, 4), 10.0, 0.25, 9),  # the kernels with the transform in registers
    ((108, 54, 12), 10.0, 0.25, None),
    ((16, 2, 1), 10.0, 0.25, None),
])
def test_incompressible_velocity(cells, h, dt, plan, monkeypatch):
    """Every inverse pass adds the kept velocity in place."""
    if plan is not None:
        monkeypatch.setenv("FHD_PLAN_XY", str(plan))
    p, _, g, o = pair(SCHEME_INCOMPRESSIBLE, cells, 7, h, 1e-3 * h ** 3, dt)
    g.step(50)
    g.sync()
    o.step(50)
    assert rel(g.velocity(), o.velocity()) < 1e-6


@pytest.mark.parametrize("dt", [2.0, 40.0])
def test_stiff_viscous_step(dt):
    """Viscous numbers of order one and above: little or nothing of the velocity is kept out of the solve, and
    the error is that of a solve of the whole velocity, 3.5e-6 over 50 steps, with the modes' 1 + x between."""
    p, _, g, o = pair(SCHEME_INCOMPRESSIBLE, (24, 32, 16), 9, 1.0, 1e-6, dt)
    g.step(50)
    g.sync()
    o.step(50)
    assert rel(g.velocity(), o.velocity()) < 1e-5


@pytest.mark.parametrize("scheme", [SCHEME_INCOMPRESSIBLE, SCHEME_QUASI_NEUTRALLY_BUOYANT])
def test_kept_velocity_stays_divergence_free(scheme):
    """1500 steps at the largest kept share (63/64)."""
    p, _, g, o = pair(scheme, (16, 16, 16), 11, 10.0, 0.1, 0.25)
    g.step(1500)
    rms = np.sqrt(np.mean(np.square(g.velocity())))
    assert g.max_divergence() * 10.0 / rms < 5 * 8.4e-7


def lattice(rng, cells, h, n):
    """n sites of a lattice of 1.25 cells, displaced by up to 0.12: pairs within the WCA range, none inside."""
    m = [int(c / 1.25) for c in cells]
    at = np.stack(np.unravel_index(rng.choice(m[0] * m[1] * m[2], n, replace=False), m), 1)
    box = np.array(cells, dtype=np.float64)
    return ((((at + 0.5) / m - 0.5) * box + rng.uniform(-0.12, 0.12, (n, 3))) * h).T.ravel()


@pytest.mark.parametrize("scheme,h,kernel", [(SCHEME_STOKES_LIMIT, 1.0, 3), (SCHEME_STOKES_LIMIT, 0.7, 4),
                                             (SCHEME_QUASI_NEUTRALLY_BUOYANT, 1.0, 3)])
def test_forces_of_close_pairs_after_100_steps(scheme, h, kernel):
    """The offset of the evaluated position is rounded once (2^-26 to 2^-25 of a cell, 1.2e-8 root mean square a
    coordinate, 2.4e-8 sigma of a pair's distance), and a pair at contact changes its force by about 25 times that
    part: 6e-7.  Bound: three times that; a run that rounds its positions at every step is ten steps' root away."""
    cells, n = (32, 24, 32), 800
    rng = np.random.default_rng(17)
    q = lattice(rng, cells, h, n)
    print(f"[gpu-case] precision forces scheme={scheme} h={h}", flush=True)
    p = make_params(scheme, cells=cells, box=tuple(h * m for m in cells), np=n, kernel_points=kernel,
                    temperature=1e-3, dt=0.05 * h * h, seed=23, initial_positions=1, wca_sigma=h,
                    cutoff=2.0 ** (1.0 / 6.0) * h)
    g, o = F.Simulation(p), O.Oracle(p)
    g.set_particles(q)
    o.set_particles(q)
    assert np.abs(g.particles() - q).max() < 2.0 ** -38 * h
    g.step(100)
    g.sync()
    o.step(100)
    e = rel(g.forces(), o.forces())
    print(f"  forces {e:.1e}, positions {np.abs(g.particles() - o.particles()).max() / h:.1e}", flush=True)
    assert e < 1.8e-6


def test_positions_resume_with_their_low_parts():
    """Positions read out and set again are the same state, in cells that are no power of two."""
    cells, h, n = (16, 24, 16), 0.3, 200
    p = make_params(SCHEME_STOKES_LIMIT, cells=cells, box=tuple(h * m for m in cells), np=n, kernel_points=3,
                    temperature=1e-3, dt=0.05, seed=5, initial_positions=0, nonbonded=0, cutoff=0.0)
    print("[gpu-case] precision resume", flush=True)
    a, b = F.Simulation(p), F.Simulation(p)
    for _ in range(6):
        q = a.particles()
        b.set_particles(q)
        assert np.array_equal(b.particles(), q)
        a.step(1)
        b.step(1)
        assert np.array_equal(a.particles(), b.particles())
