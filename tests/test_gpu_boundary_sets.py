"""The ghost passes in one launch (boundary_kernel) and inside the step kernel, over the boundary sets
whose passes read each other's ghosts: closed next to closed, closed next to a copied periodic plane,
closed next to inflow, edges and corners, the smallest grid, planes of one, just over one and several
blocks, each contiguous axis.

Against the oracle in FP64, from an equilibrium start (whose two boundary passes run the kernel on
their own) and from a record.  The passes copy values; the collision and the inflow ghosts round a few
units in the last place of populations below 0.35 (2^-54) a step: 10 steps * 8 * 2^-54 = 4.4e-15,
taken as 2e-14.
"""
import numpy as np
import pytest

import oracle
from lbm_amd.domain import Domain

pytestmark = pytest.mark.gpu

SETS = [(1, 11, 12), (1, 22, 11), (22, 11, 12), (11, 21, 22), (0, 11, 22), (11, 0, 22), (21, 12, 0), (22, 22, 22),
        (1, 21, 0), (1, 0, 12), (0, 0, 21)]
DIMS = [(2, 3, 2), (8, 8, 8), (5, 17, 16), (33, 9, 30)]


@pytest.mark.parametrize("fold", ["1", "0"])
@pytest.mark.parametrize("bnd", SETS)
@pytest.mark.parametrize("q", [19, 27])
def test_boundary_sets_match_oracle(monkeypatch, q, bnd, fold):
    monkeypatch.setenv("LBM_FOLD", fold)
    o = dict(ibgk=3, ihrr=1, ivreman=1, smagorinsky=0.17, kinevisc=0.02, ibnd=bnd[0], jbnd=bnd[1], kbnd=bnd[2])
    uini, udir = (0.04, 20.0) if bnd[0] == 1 else (0.0, 0.0)
    for d, dims in enumerate(DIMS):
        monkeypatch.setenv("LBM_FAST_AXIS", str(d % 3))
        print(f"D3Q{q} {bnd} {dims} fold={fold}", flush=True)
        shape = tuple(n + 2 for n in reversed(dims))
        rng = np.random.default_rng(d)
        mom = [1.0 + 0.01 * rng.random(shape)] + [0.03 * rng.random(shape) for _ in range(3)]
        sim = oracle.OracleSim(q, dims, "f64", **o)
        sim.init_equilibrium(*mom, uini=uini, udir=udir)
        with Domain(q, dims, "f64", iturb_pos=1, **o) as dom:
            dom.set_inflow(uini, udir)
            dom.init_equilibrium(*mom)
            assert np.abs(dom.get_state() - sim.f1).max() < 2e-14
            dom.step(0, 5)
            sim.run(0, 5, uini=uini, udir=udir)
            f = sim.f1.copy()
            assert np.abs(dom.get_state() - f).max() < 2e-14
            dom.set_state(f)
            sim.restart(f)
            dom.step(5, 5)
            sim.run(5, 10, uini=uini, udir=udir)
            assert np.abs(dom.get_state() - sim.f1).max() < 2e-14
