"""Spreading inside the forward xy transform (plane_spread.h) at the edges of its dispatch, against
the FP64 oracle: planes with more sources than its list holds (6144, taken in chunks), nodes shared
by more than 255 sources (two 32-bit sums), force and thermal drift in one row, RFD pairs in both
modes and with a displacement that crosses cells, boxes narrower than a stencil, planes of every
workgroup class of the runtime-size kernels.

Tolerances: those of the trajectory tests (FP32 fields against FP64: positions 1e-5, velocities
1e-4; an RFD pair's difference of weights 1e-3 apart is good to about 6e-8 / 1e-3 of itself)."""
import numpy as np
import pytest

import fluam_amd as F
import oracle_lib as O
from fluam_amd._abi import make_params, SCHEME_STOKES_LIMIT, SCHEME_QUASI_NEUTRALLY_BUOYANT

pytestmark = pytest.mark.gpu
ST, QNB = SCHEME_STOKES_LIMIT, SCHEME_QUASI_NEUTRALLY_BUOYANT


def rel(a, b):
    return np.linalg.norm(a - b) / max(np.linalg.norm(b), 1e-300)


@pytest.mark.parametrize("scheme,cells,n,kernel,kw", [
    (ST, (32, 32, 16), 600, 4, {}),
    (ST, (16, 16, 8), 20000, 4, {}),
    (QNB, (16, 16, 8), 20000, 3, {}),
    (QNB, (32, 16, 24), 30000, 4, {}),
    (ST, (64, 64, 8), 30000, 3, {}),
    (ST, (8, 4, 2), 5, 4, {}),
    (QNB, (8, 4, 2), 5, 3, {}),
    (ST, (4, 8, 16), 7, 3, {"rfd_mode": 1}),
    (ST, (24, 32, 16), 400, 4, {"rfd_mode": 1}),
    (ST, (24, 32, 16), 400, 4, {"rfd_delta": 0.2}),
    (QNB, (108, 36, 12), 500, 4, {}),
    (ST, (72, 108, 8), 700, 3, {}),
    (ST, (128, 72, 8), 700, 4, {}),
    (QNB, (36, 48, 8), 400, 3, {"mass": 2.0}),
    # more particles than the interpolation keeps all rows of in flight (32768)
    (ST, (32, 16, 16), 33000, 4, {}),
    (QNB, (24, 24, 16), 33000, 3, {}),
])
def test_plane_spread_matches_oracle(scheme, cells, n, kernel, kw):
    print(f"[gpu-case] plane spread scheme={scheme} cells={cells} np={n} k={kernel} {kw}", flush=True)
    p = make_params(scheme, cells=cells, np=n, kernel_points=kernel, nonbonded=0, temperature=1e-3, dt=0.05,
                    seed=61 + n, initial_positions=0, cutoff=0.0, **kw)
    g, o = F.Simulation(p), O.Oracle(p)
    q0 = o.particles()
    g.step(3)
    g.sync()
    o.step(3)
    qg, qo = g.particles(), o.particles()
    assert rel(qg, qo) < 1e-5
    assert rel(qg - q0, qo - q0) < 1e-3
    assert rel(g.velocity(), o.velocity()) < 1e-4


def test_plane_spread_is_deterministic_when_crowded():
    p = make_params(ST, cells=(16, 16, 8), np=20000, kernel_points=4, nonbonded=0, temperature=1e-3, dt=0.05, seed=5,
                    initial_positions=0, cutoff=0.0)
    runs = []
    for _ in range(2):
        s = F.Simulation(p)
        s.step(3)
        runs.append((s.velocity(), s.particles()))
    assert np.array_equal(runs[0][0], runs[1][0]) and np.array_equal(runs[0][1], runs[1][1])
