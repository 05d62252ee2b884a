"""The W kernel of fluid.hip (explicit right-hand side with its stochastic stress) over boxes that its
16 x 16 x chunk cell blocks do not divide, against the FP64 oracle: both solves of an incompressible
step (the second starts from the terms it shares with the first) and the inertial scheme's single one."""
import numpy as np
import pytest

import fluam_amd as F
import oracle_lib as O
from fluam_amd._abi import make_params, SCHEME_INCOMPRESSIBLE, SCHEME_QUASI_NEUTRALLY_BUOYANT

pytestmark = pytest.mark.gpu


def rel(a, b):
    return np.linalg.norm(a - b) / max(np.linalg.norm(b), 1e-300)


# A step's velocity is held in FP32: relative L2 below 1e-5 of the oracle's, as for the other parts of
# a step (1e-4 with particles).
@pytest.mark.parametrize("chunk", [1, 2, 4])
@pytest.mark.parametrize("cells", [(2, 1, 1), (6, 3, 2), (18, 27, 9), (16, 16, 6), (32, 16, 27)])
def test_w_pass_matches_oracle(cells, chunk, monkeypatch):
    print(f"[gpu-case] W pass {cells} chunk {chunk}", flush=True)
    monkeypatch.setenv("FHD_ZCHUNK", str(chunk))
    p = make_params(SCHEME_INCOMPRESSIBLE, cells=cells, temperature=1e-2, dt=0.1, seed=9, background=(0.02, -0.01, 0.03))
    g, o = F.Simulation(p), O.Oracle(p)
    g.step(4)
    g.sync()
    o.step(4)
    assert rel(g.velocity(), o.velocity()) < 1e-5


@pytest.mark.parametrize("chunk", [1, 2, 4])
def test_w_pass_of_the_inertial_scheme(chunk, monkeypatch):
    print(f"[gpu-case] W pass inertial chunk {chunk}", flush=True)
    monkeypatch.setenv("FHD_ZCHUNK", str(chunk))
    p = make_params(SCHEME_QUASI_NEUTRALLY_BUOYANT, cells=(24, 12, 6), np=20, kernel_points=3, temperature=1e-3,
                    dt=0.05, seed=3, initial_positions=1, cutoff=0.0)
    g, o = F.Simulation(p), O.Oracle(p)
    g.step(4)
    g.sync()
    o.step(4)
    assert rel(g.velocity(), o.velocity()) < 1e-4
