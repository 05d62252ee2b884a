"""fhd_bytes_needed, the figure that the serving loop admits jobs by, is what fhd_create allocates."""
import pytest

import fluam_amd as F
from fluam_amd._abi import (make_params, SCHEME_INCOMPRESSIBLE, SCHEME_STOKES_LIMIT,
                            SCHEME_QUASI_NEUTRALLY_BUOYANT)

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("scheme,kw", [
    (SCHEME_INCOMPRESSIBLE, {}),
    (SCHEME_STOKES_LIMIT, {}),
    (SCHEME_STOKES_LIMIT, {"np": 1000000}),
    (SCHEME_STOKES_LIMIT, {"np": 1000000, "cutoff": 1.1}),
    (SCHEME_QUASI_NEUTRALLY_BUOYANT, {}),
    (SCHEME_QUASI_NEUTRALLY_BUOYANT, {"np": 500000, "mass": 2.0}),
])
def test_bytes_needed_is_what_a_context_takes(scheme, kw):
    """To 2% and 2 MiB (the allocator's granule) for each of the ten largest buffers."""
    print(f"[gpu-case] bytes needed scheme={scheme} {kw}", flush=True)
    kw = {"cutoff": 0.0, **kw}
    p = make_params(scheme, cells=(128, 128, 256), temperature=1e-3, dt=0.05, seed=1, kernel_points=4,
                    initial_positions=0, nonbonded=int(kw["cutoff"] > 0), wca_sigma=1.0, **kw)
    F.Simulation(make_params(SCHEME_INCOMPRESSIBLE, cells=(16, 16, 16), temperature=1e-3, dt=0.05)).step(1)
    before = F.mem_info()[0]
    s = F.Simulation(p)
    used = before - F.mem_info()[0]
    need = F.bytes_needed(p)
    del s
    print(f"  needed {need / 2 ** 20:.1f} MiB, used {used / 2 ** 20:.1f} MiB", flush=True)
    assert abs(need - used) < 0.02 * used + 20 * 2 ** 20
