"""The 32-bit sums of the spreading (plane_spread.h) at the edges of their bounds, against the FP64 oracle:
boxes narrower than a stencil, whose nodes take several weights of one source, and cells so flat that a random
displacement leaves the neighbouring columns.  Forces come from springs to fixed points, so vector values,
thermal drift, RFD pairs and the excess-mass impulses are all of the size that sets the scale.

Tolerances: those of the trajectory tests (FP32 fields against FP64: displacements 1e-3, velocities 1e-4), and
where the result vanishes (in the narrowest boxes the projection leaves nothing of a Stokes field, and a 4-point
stencil of two nodes sees the mean alone) what 32 bits round: a position's offset by 2^-25 of a cell in each of a
step's two updates, a velocity by 1e-6 of what the force on one cell would give."""
import numpy as np
import pytest

import fluam_amd as F
import oracle_lib as O
from fluam_amd._abi import make_params, SCHEME_STOKES_LIMIT, SCHEME_QUASI_NEUTRALLY_BUOYANT

pytestmark = pytest.mark.gpu
ST, QNB = SCHEME_STOKES_LIMIT, SCHEME_QUASI_NEUTRALLY_BUOYANT


def near(a, b, rel, each):
    """|a - b| within `rel` of |b| and `each` a value."""
    assert np.linalg.norm(a - b) <= rel * np.linalg.norm(b) + each * np.sqrt(b.size)


def trapped(path, q, k, rng):
    """A spring file that pulls particle i with a force of about k[i] (springs k[i] of rest length 0 to points at
    a distance of about 1)."""
    x = q.reshape(3, -1).T + rng.normal(0.0, 0.6, (q.size // 3, 3))
    lines = ["0", str(len(x))] + [f"{i} {k[i]} 0.0 {a!r} {b!r} {c!r}" for i, (a, b, c) in enumerate(x.tolist())]
    path.write_text("\n".join(lines) + "\n")
    return str(path)


def run(tmp_path, scheme, cells, n, kernel, seed, k=0.01, box=None, steps=3, **kw):
    print(f"[gpu-case] spread bounds scheme={scheme} cells={cells} np={n} k={kernel} seed={seed} {kw}", flush=True)
    rng = np.random.default_rng(seed)
    box = tuple(float(m) for m in cells) if box is None else box
    q = (rng.uniform(-0.5, 0.5, (n, 3)) * np.array(box)).T.ravel()
    bonds = trapped(tmp_path / "traps.dat", q, np.full(n, k), rng)
    p = make_params(scheme, cells=cells, box=box, np=n, kernel_points=kernel, nonbonded=0, temperature=1e-3, dt=0.05,
                    seed=seed, initial_positions=0, cutoff=0.0, bonded_forces=bonds, **kw)
    g, o = F.Simulation(p), O.Oracle(p)
    g.set_particles(q)
    o.set_particles(q)
    g.step(steps)
    g.sync()
    o.step(steps)
    h = [l / m for l, m in zip(box, cells)]
    unit = 1e-6 * np.abs(o.forces()).max() * max(h) ** 2 / (p.shearviscosity * h[0] * h[1] * h[2])
    near(g.particles() - q, o.particles() - q, 1e-3, 2 * steps * 2.0 ** -25 * max(h))
    near(g.velocity(), o.velocity(), 1e-4, unit)
    near(g.particle_velocities(), o.particle_velocities(), 1e-3, unit)


NARROW = [(16, 1, 1), (2, 1, 1), (2, 2, 2), (4, 1, 2), (8, 2, 1), (16, 16, 1), (16, 8, 1), (16, 1, 8), (6, 3, 3), (2, 8, 4)]


@pytest.mark.parametrize("kernel", [3, 4])
@pytest.mark.parametrize("cells", NARROW)
@pytest.mark.parametrize("scheme,n,kw", [(QNB, 1, {}), (QNB, 3, {}), (QNB, 40, {"mass": 2.0}), (ST, 1, {}), (ST, 3, {}), (ST, 40, {})])
def test_boxes_narrower_than_a_stencil(tmp_path, scheme, n, kw, cells, kernel):
    for seed in range(3):
        run(tmp_path, scheme, cells, n, kernel, 100 * n + seed, **kw)


def test_one_axis_of_one_cell_without_forces(tmp_path):
    """Thermal drift alone sets the scale."""
    for seed in range(8):
        run(tmp_path, QNB, (16, 1, 1), 1, 4, 40 + seed, k=0.0)


@pytest.mark.parametrize("kernel", [3, 4])
def test_displacements_across_flat_cells(tmp_path, kernel):
    """Displacements of up to 1.45 in cells of 0.25 x 0.25 x 2."""
    run(tmp_path, ST, (32, 24, 8), 500, kernel, 9, box=(8.0, 6.0, 16.0), rfd_delta=0.5)
