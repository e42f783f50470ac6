"""Totals and the solid mask for each contiguous axis, rows of less than, of and of more than a word of the mask.

Totals are FP64 sums of nx*ny*nz*q populations below 0.35 in any order: within that number times 2^-53 of numpy's, which
is below 2e-11 here.  A run with a mask does the same arithmetic for each contiguous axis: 4 steps within 4 * 8 units
in the last place of a population below 0.5 (1.8e-15), taken as 4e-15.
"""
import numpy as np
import pytest

from lbm_amd.domain import Domain
from lbm_amd.lattice import lattice

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dims", [(5, 3, 2), (31, 32, 33), (64, 7, 65), (9, 40, 70)])
@pytest.mark.parametrize("q", [19, 27])
def test_totals_and_masks(monkeypatch, q, dims):
    nx, ny, nz = dims
    rng = np.random.default_rng(q + nx)
    lat = lattice(q)
    f0 = lat.w * (1.0 + 0.05 * rng.uniform(-1, 1, (nz + 2, ny + 2, nx + 2, q)))
    mask = (rng.random(f0.shape[:3]) < 0.2).astype(np.uint8) * 3
    inner = f0[1:-1, 1:-1, 1:-1]
    want = [inner.sum()] + [(inner * c).sum() for c in (lat.cx, lat.cy, lat.cz)]
    out = []
    for axis in (0, 1, 2):
        print(f"D3Q{q} {dims}, contiguous axis {axis}", flush=True)
        monkeypatch.setenv("LBM_FAST_AXIS", str(axis))
        with Domain(q, dims, "f64", ibgk=3, ihrr=1, ivreman=1, smagorinsky=0.17, kinevisc=0.02, ibnd=0, jbnd=0, kbnd=0) as d:
            d.set_state(f0)
            for noalloc in (False, True):
                m, p = d.totals(noalloc=noalloc)
                assert np.abs(np.array([m, *p]) - want).max() < inner.size * 2.0 ** -53
            d.set_blanking(mask)
            d.step(1, 4)
            out.append(d.get_state())
    assert np.isfinite(out[0]).all()
    for o in out[1:]:
        assert np.abs(o - out[0]).max() < 4e-15
