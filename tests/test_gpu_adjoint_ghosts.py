"""The states that the reverse sweep recomputes (lbm_adjoint_run): with a checkpoint before every step
nothing is recomputed, so any other spacing has to give the same objective and gradients bit for bit, if
each recomputed step finds the ghosts that the forward step found (ghost_keep_kernel).  Every boundary
set the adjoint takes, each contiguous axis, the smallest grid among them.
"""
import numpy as np
import pytest

from lbm_amd.domain import Domain

pytestmark = pytest.mark.gpu

SETS = [(1, 0, 12), (1, 22, 0), (1, 0, 0), (0, 0, 11), (0, 21, 0), (12, 0, 0)]


@pytest.mark.parametrize("fold", ["1", "0"])
@pytest.mark.parametrize("bnd", SETS)
@pytest.mark.parametrize("q", [19, 27])
def test_recomputed_states_are_the_forward_ones(monkeypatch, q, bnd, fold):
    monkeypatch.setenv("LBM_FOLD", fold)
    for n, dims in enumerate([(2, 3, 2), (9, 8, 7), (12, 66, 5)]):
        monkeypatch.setenv("LBM_FAST_AXIS", str(n))
        print(f"D3Q{q} {bnd} {dims} fold={fold}", flush=True)
        shape = tuple(x + 2 for x in reversed(dims))
        rng = np.random.default_rng(n)
        mom = [1.0 + 0.01 * rng.random(shape)] + [0.03 * rng.random(shape) for _ in range(3)]
        force = 1e-4 * rng.random(shape + (3,))
        got = []
        for every in (1, 3, 8):
            with Domain(q, dims, "f64" if n == 1 else "f32", ibgk=3, ihrr=1, ivreman=1, smagorinsky=0.17, kinevisc=0.02,
                        iturb_pos=1, ibnd=bnd[0], jbnd=bnd[1], kbnd=bnd[2]) as d:
                d.set_inflow(0.04, 10.0)
                d.init_equilibrium(*mom)
                d.set_external_forcing(force)
                d.step(0, 3)
                got.append([np.asarray(a) for a in d.adjoint(3, 8, every, tuple((1, x) for x in dims))])
        assert np.abs(got[0][1]).max() > 0
        for other in got[1:]:
            for a, b in zip(got[0], other):
                assert a.tobytes() == b.tobytes()
