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


@pytest.mark.parametrize("scheme,cells,n,kernel,kw", [
    (ST, (32, 32, 16), 600, 4, {}),    # one 32-bit sum
    (ST, (16, 16, 8), 5000, 4, {}),    # two sums, more hits than the list holds
    (ST, (16, 16, 8), 20000, 3, {}),   # two sums, not listed
    (QNB, (32, 32, 16), 600, 3, {}),
    (QNB, (16, 16, 8), 5000, 3, {}),
    (QNB, (16, 16, 8), 20000, 4, {}),
    (QNB, (8, 4, 2), 300, 4, {}),      # two sums in a box narrower than a stencil
    (ST, (64, 16, 8), 9000, 4, {"rfd_delta": 2.5}),  # displaced beyond the neighbouring blocks: one scale
    (ST, (72, 36, 8), 9000, 4, {}),    # runtime-size passes
    (QNB, (128, 128, 4), 12000, 4, {}),
    (ST, (64, 64, 16), 140000, 4, {}),
    (QNB, (48, 24, 16), 140000, 3, {}),
])
def test_crowded_planes_with_forces(tmp_path, scheme, cells, n, kernel, kw):
    run(tmp_path, scheme, cells, n, kernel, 300 + kernel, **kw)


@pytest.mark.parametrize("mode", [0, 2])
def test_crowded_replicas_equal_alone(mode):
    """Planes without a list, in boxes that a merged batch gives to the runtime-size passes."""
    ps = [make_params(ST, cells=c, np=n, kernel_points=k, nonbonded=0, temperature=1e-3, dt=0.05, seed=40 + n,
                      initial_positions=0, cutoff=0.0)
          for c, n, k in (((16, 16, 16), 9000, 4), ((32, 16, 24), 14000, 3), ((32, 32, 32), 40, 4), ((64, 64, 16), 30000, 4))]
    print(f"[gpu-case] crowded replicas mode={mode}", flush=True)
    b = F.Batch(ps)
    b.set_mode(mode)
    b.step(3)
    b.sync()
    for p, r in zip(ps, b.replicas):
        alone = F.Simulation(p)
        alone.step(3)
        assert np.array_equal(alone.velocity(), r.velocity())
        assert np.array_equal(alone.particles(), r.particles())
    b.close()


def test_weak_forces_beside_a_strong_one(tmp_path):
    """Thirty particles feel a force a millionth of that on one particle of the same plane, which sixty force-free ones
    surround (so many sources in reach of a node take bits from its sum).  The Stokes flow is linear: what the
    weak forces add to their particles' velocities is what they give alone, up to the rounding of the strong
    one's field, about 2e-7 of its root mean square in each of the two runs subtracted; bound: three times that."""
    m, rng = 128, np.random.default_rng(4)
    q = np.zeros((91, 3))
    q[1:61] = rng.uniform(-1.5, 1.5, (60, 3))
    q[61:] = np.stack([*rng.uniform(12.0, 52.0, (2, 30)) * rng.choice([-1.0, 1.0], (2, 30)), rng.uniform(-0.5, 0.5, 30)], 1)
    q += 0.3
    pull = rng.standard_normal((91, 3))
    pull /= np.linalg.norm(pull, axis=1)[:, None]

    def velocities(name, strong, weak):
        k = {**({0: 1.0} if strong else {}), **({i: 1e-6 for i in range(61, 91)} if weak else {})}
        lines = ["0", str(len(k))] + [f"{i} {c} 0.0 " + " ".join(repr(float(x)) for x in q[i] + pull[i]) for i, c in k.items()]
        (tmp_path / name).write_text("\n".join(lines) + "\n")
        p = make_params(ST, cells=(m, m, m), np=91, kernel_points=4, nonbonded=0, temperature=0.0, dt=1e-4, seed=1,
                        initial_positions=0, cutoff=0.0, bonded_forces=str(tmp_path / name))
        print(f"[gpu-case] weak beside strong: {name}", flush=True)
        g = F.Simulation(p)
        g.set_particles(q.T.ravel())
        g.step(1)
        return g.particle_velocities().reshape(3, -1)[:, 61:], np.sqrt(np.mean(np.square(g.velocity())))

    strong, rms = velocities("strong", True, False)
    both, _ = velocities("both", True, True)
    alone, _ = velocities("weak", False, True)
    off = np.sqrt(np.mean(np.square(both - strong - alone)))
    print(f"  off {off:.2e} of {np.sqrt(np.mean(np.square(alone))):.2e}, rms {rms:.2e}", flush=True)
    assert off < 3.0 * np.sqrt(2.0) * 2e-7 * rms
