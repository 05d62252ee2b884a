"""The z pass of fft_z.hip (column lengths that are a product of two radices): each length's transforms
in both directions against numpy, and the solve against the FP64 oracle at the column-tile widths of a
workgroup, with tiles of unequal width and workgroup counts that do not divide among the eight XCDs."""
import numpy as np
import pytest

import fluam_amd as F
import oracle_lib as O
from fluam_amd._abi import make_params, SCHEME_INCOMPRESSIBLE, SCHEME_STOKES_LIMIT

pytestmark = pytest.mark.gpu


def rel(a, b):
    return np.linalg.norm(a - b) / max(np.linalg.norm(b), 1e-300)


# FP32 transforms of n points are off by about log2(n) 2^-24 relative to the largest mode, below
# 2e-6 here; the bound is 1e-5.
@pytest.mark.parametrize("mz", [16, 18, 24, 27, 32, 36, 48, 54, 64, 72, 81, 96, 108, 128, 144, 192, 256])
def test_z_lengths_match_numpy(mz):
    shape = (mz, 3, 54)  # 28 columns: one tile of the one-component transform is narrower
    print(f"[gpu-case] z pass {shape}", flush=True)
    rng = np.random.default_rng(mz)
    a = rng.standard_normal(shape)
    got = F.fft_r2c(a)
    ref = np.fft.rfftn(a)
    assert np.abs(got - ref).max() < 1e-5 * np.abs(ref).max()
    back = F.fft_c2r(ref, shape[2])
    assert np.abs(back - a * a.size).max() < 1e-5 * np.abs(a * a.size).max()


# (mx, my, mz): the smallest box of one column tile, tiles that all differ from the rest by one
# column, one row more than the XCDs divide, the longest two-radix column.  A step's velocity is held
# in FP32: relative L2 below 1e-5 of the oracle's, as for the other FFT paths.
@pytest.mark.parametrize("tile", [2, 4, 8, 16])
@pytest.mark.parametrize("cells,scheme", [((2, 1, 16), SCHEME_INCOMPRESSIBLE), ((18, 3, 27), SCHEME_INCOMPRESSIBLE),
                                          ((16, 12, 72), SCHEME_INCOMPRESSIBLE), ((16, 12, 72), SCHEME_STOKES_LIMIT),
                                          ((6, 4, 256), SCHEME_INCOMPRESSIBLE), ((6, 4, 256), SCHEME_STOKES_LIMIT)])
def test_z_solve_matches_oracle(cells, tile, scheme, monkeypatch):
    print(f"[gpu-case] z solve {cells} tile {tile} scheme {scheme}", flush=True)
    monkeypatch.setenv("FHD_BTILE", str(tile))
    if scheme == SCHEME_STOKES_LIMIT:
        p = make_params(scheme, cells=cells, np=5, initial_positions=1, temperature=1e-2, dt=0.05, seed=5,
                        kernel_points=4, cutoff=0.0)
    else:
        p = make_params(scheme, cells=cells, temperature=1e-2, dt=0.1, seed=5)
    g, o = F.Simulation(p), O.Oracle(p)
    g.step(3)
    g.sync()
    o.step(3)
    assert rel(g.velocity(), o.velocity()) < 1e-5 * (10 if p.np else 1)
    assert g.max_divergence() < 1e-6
