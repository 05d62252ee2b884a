"""The schedule is a rule on the grid's shape: a run's bits depend on nothing that was timed, and what
fhd_get_schedule reports is what runs."""
import numpy as np
import pytest

import fluam_amd as F
from fluam_amd._abi import make_params, SCHEME_INCOMPRESSIBLE, SCHEME_STOKES_LIMIT

pytestmark = pytest.mark.gpu


def sim(cells, np_=0):
    print(f"[gpu-case] schedule cells={cells} np={np_}", flush=True)
    if np_ == 0:
        return F.Simulation(make_params(SCHEME_INCOMPRESSIBLE, cells=cells, temperature=1e-3, dt=0.05, seed=5))
    return F.Simulation(make_params(SCHEME_STOKES_LIMIT, cells=cells, np=np_, kernel_points=4, nonbonded=0,
                                    temperature=1e-3, dt=0.05, seed=5, initial_positions=0, cutoff=0.0))


@pytest.mark.parametrize("cells,np_", [((96, 96, 8), 0), ((128, 128, 8), 0), ((128, 128, 8), 60), ((48, 48, 24), 60)])
def test_no_timing_chooses_a_runs_bits(cells, np_, monkeypatch):
    monkeypatch.setenv("FHD_AUTOTUNE", "0")
    a = sim(cells, np_)
    monkeypatch.setenv("FHD_AUTOTUNE", "1")
    b = sim(cells, np_)
    assert a.schedule() == b.schedule()
    a.step(4)
    b.step(4)
    assert np.array_equal(a.velocity(), b.velocity())
    if np_:
        assert np.array_equal(a.particles(), b.particles())


def test_the_schedule_in_use_is_reported(monkeypatch):
    monkeypatch.setenv("FHD_BTILE", "16")
    monkeypatch.setenv("FHD_ZCHUNK", "16")
    s = sim((32, 32, 32)).schedule()
    assert (s["z_column_tile"], s["w_z_chunk"], s["w_z_chunk_batched"]) == (8, 4, 4)
    assert sim((32, 32, 12)).schedule()["z_column_tile"] == 16  # a length of the runtime-size z pass
    monkeypatch.setenv("FHD_ZCHUNK", "3")
    monkeypatch.setenv("FHD_PLAN_XY", "5")
    s = sim((128, 128, 4)).schedule()
    assert (s["xy_radix_plan"], s["xy_radix_plan_inverse"], s["w_z_chunk"]) == (5, 5, 2)
    s = sim((128, 128, 4), 20).schedule()  # spreading has one plan
    assert (s["xy_radix_plan"], s["xy_radix_plan_inverse"]) == (2, 5)
    s = sim((48, 48, 24)).schedule()  # no other plans
    assert (s["xy_radix_plan"], s["xy_radix_plan_inverse"]) == (0, 0)
