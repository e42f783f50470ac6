"""The deposit of the actuator points in lists per block (turbine_deposit_kernel) and the lookup of the
airfoil tables by all threads: more points than a list's 256 entries, points whose stencils reach over
the grid's edges or lie outside it, rotors that overlap, tables of 2 rows, of 300 (more than the
block's threads) and without the angle, against the oracle in FP64.

The forces are sums of up to 20 deposits and enter the populations as differences below 1e-3: 6 steps
of a few units in the last place of populations below 0.35 (2^-54) and 20 * 2^-53 relative of 1e-3:
below 6 * (8 * 2^-54 + 20 * 2^-53 * 1e-3) = 3e-15, taken as 2e-14.
"""
import numpy as np
import pytest

import oracle
from lbm_amd.domain import Domain

pytestmark = pytest.mark.gpu


def rotors(n, dims, rows, seed):
    rng = np.random.default_rng(seed)
    nx, ny, nz = dims
    hub = np.stack([rng.uniform(-3, nx + 4, n), rng.uniform(1, ny, n), rng.uniform(1, nz, n)], 1)
    hub[0] = (nx / 2, ny / 2, nz / 2)
    lo, hi = (-180.0, 180.0) if rows > 2 else (170.0, 171.0)
    deg = np.linspace(lo, hi, rows)
    foil = np.stack([deg, np.sin(np.deg2rad(2 * deg)), 0.02 + np.sin(np.deg2rad(deg)) ** 2], 1)
    nc = 17
    return dict(hub=hub, yaw=rng.uniform(-0.3, 0.3, n), tilt=rng.uniform(-0.1, 0.1, n), omegand=np.full(n, 0.02),
                pitch=np.zeros(n), theta=rng.uniform(0, 2, n), relm=np.linspace(0.5, 6.0, nc), dc=np.full(nc, 0.3),
                chord=np.full(nc, 0.2), twist=np.linspace(13, 0, nc), nfoil=np.ones(nc, np.int32), foils=[foil], nblades=3)


@pytest.mark.parametrize("axis", ["0", "1", "2"])
@pytest.mark.parametrize("n,rows", [(1, 2), (1, 73), (6, 300)])
def test_deposit_matches_oracle(monkeypatch, axis, n, rows):
    monkeypatch.setenv("LBM_FAST_AXIS", axis)
    dims = (24, 70, 18)
    print(f"{n} rotors, {rows} rows, contiguous axis {axis}", flush=True)
    o = dict(ibgk=3, ihrr=1, ivreman=1, smagorinsky=0.17, kinevisc=0.01, ibnd=1, jbnd=0, kbnd=12)
    shape = tuple(m + 2 for m in reversed(dims))
    rng = np.random.default_rng(3)
    mom = [np.ones(shape), 0.05 + 0.01 * rng.random(shape)] + [0.01 * rng.random(shape) for _ in range(2)]
    t = rotors(n, dims, rows, 7)
    sim = oracle.OracleSim(19, dims, "f64", **o)
    sim.init_equilibrium(*mom, uini=0.05)
    T = dict(t, xhub=t["hub"][:, 0], yhub=t["hub"][:, 1], zhub=t["hub"][:, 2], theta=t["theta"].copy())
    sim.run(0, 6, uini=0.05, turbines=T)
    with Domain(19, dims, "f64", **o) as d:
        d.set_inflow(0.05)
        d.set_turbines(t)
        d.init_equilibrium(*mom)
        d.step(0, 6)
        assert np.abs(d.get_state() - sim.f1).max() < 2e-14
        assert np.abs(d.turbine_theta() - T["theta"]).max() < 1e-14
