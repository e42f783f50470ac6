"""The turbulence generator (lbm_generate_turbulence) where its chain of slices changes form: values kept in
registers, two more a thread for every 2048 cells of a slice, up to 16384, in memory beyond.  Sizes at and
just past those edges, odd ones, the smallest slice and a single window step, against the numpy oracle.

Tolerances as of the transforms and the chain elsewhere: 1e-9 in FP64 (direct sums of at most 129 terms of
order 1, normalized to deviation 1), 2e-4 in FP32 (the recursion and the normalization run in FP32).
"""
import numpy as np
import pytest

import pseudo2d
from lbm_amd.domain import Domain

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("storage,tol", [("f64", 1e-9), ("f32", 2e-4)])
@pytest.mark.parametrize("ny,nz,nrturb", [(2, 3, 2), (64, 32, 3), (41, 50, 3), (64, 64, 1), (63, 66, 2), (126, 65, 3),
                                          (128, 128, 2), (127, 129, 2), (128, 129, 2)])
def test_slice_sizes_match_oracle(storage, tol, ny, nz, nrturb):
    print(f"turbulence {storage} {ny}x{nz} nrturb={nrturb}", flush=True)
    with Domain(19, (16, ny, nz), storage, ibgk=3, ihrr=1, ivreman=1, smagorinsky=0.17, kinevisc=1e-3, ibnd=1, kbnd=12) as d:
        got = d.generate_turbulence(nrturb, 1e-3, 7)
        again = d.generate_turbulence(nrturb, 1e-3, 7)
    ref = pseudo2d.generate(ny, nz, nrturb, 7)
    for g, a, r in zip(got, again, ref):
        assert g.tobytes() == a.tobytes()
        err = np.abs(g.astype(np.float64) - r).max()
        print(f"  max |diff| {err:.3e}", flush=True)
        assert err <= tol
