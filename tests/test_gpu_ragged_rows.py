"""Rows whose length is no multiple of 64 bytes or of a wavefront: the step kernel's lanes past the
end of a row store copies of its last cell into the padding (Layout::row_store_end), next to the
wrapped neighbours, the folded faces, the inflow planes, the solid mask and the averaging sums.

Against the oracle in the storage's precision, with every input on.  Bounds, fixed before the first
run: the oracle and the kernels round each of the 12 steps differently by a few units in the last
place of populations below 0.35 (2^-25 resp. 2^-54 each), and the collision does not amplify them:
12 * 4 * 2^-25 = 1.4e-6 in FP32, 2.7e-15 in FP64, taken as 2e-6 and 1e-14.  The averages' means are
sums of 5 such steps' velocities (bounds times 8: three times 9 of 27 populations enter a velocity).
"""
import numpy as np
import pytest

import oracle
from lbm_amd import inputs
from lbm_amd.domain import Domain

pytestmark = pytest.mark.gpu

# contiguous lengths: one cell more and less than 64 and 128 bytes, the wavefront, and two cells
LENGTHS = {"f32": (2, 15, 16, 17, 31, 33, 63, 65), "f64": (7, 8, 9, 17, 63, 66)}


@pytest.mark.parametrize("q", [19, 27])
@pytest.mark.parametrize("storage,n0", [(s, n) for s in LENGTHS for n in LENGTHS[s]])
def test_row_lengths_match_oracle(storage, n0, q):
    dims = (24, n0, 7)                     # j periodic: contiguous
    dt = np.float64 if storage == "f64" else np.float32
    o = dict(ibgk=3, ihrr=1, ivreman=1, smagorinsky=float(dt(0.17)), kinevisc=float(dt(0.01)), ibnd=1, jbnd=0, kbnd=12)
    print(f"rows of {n0}, D3Q{q} {storage}", flush=True)
    f0 = inputs.perturbed_uniform_flow(q, dims, seed=n0, u0=(0.05, 0, 0), order=3, dtype=dt)
    tu = inputs.turbulence_fields(3, n0, dims[2], 20, dtype=dt)
    mask = inputs.box_mask(dims, (8, max(1, n0 - 1), 1), (12, n0, 4))
    sim = oracle.OracleSim(q, dims, storage, **o)
    sim.restart(f0)
    run = dict(uini=float(dt(0.05)), blank=mask, turb=(tu[0], tu[1], tu[2], 20, float(dt(1e-3))))
    with Domain(q, dims, storage, **o) as d:
        d.set_state(f0)
        d.set_inflow(0.05)
        d.set_blanking(mask)
        d.set_turbulence(tu[0], tu[1], tu[2], 20, 1e-3)
        d.step(1, 7)
        sim.run(1, 8, **run)
        d.set_averaging(True)
        d.step(8, 5)
        sums = np.zeros((3,) + d.shape_cell)
        for it in range(8, 13):
            sim.run(it, it + 1, **run)
            sums += np.stack(sim.macros()[1:]).astype(np.float64)
        tol = 1e-14 if storage == "f64" else 2e-6
        assert np.abs(d.get_state().astype(np.float64) - sim.f1).max() < tol
        inner = (slice(1, -1),) * 3
        for got, want in zip(d.averages()[:3], sums / 5):
            assert np.abs(got[inner] - want[inner]).max() < 8 * tol
