"""The inflow/outflow planes of a duct (two closed axes) written by the step kernel but for their rows along the
walls: bit for bit the state of the separate launch, for each storage, from planes that are nothing but
those rows (2 x 2 cells) on, each contiguous axis, on both sides of the size from which it is the default.
"""
import numpy as np
import pytest

from lbm_amd.domain import Domain

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("storage", ["f32", "f64", "f16s"])
@pytest.mark.parametrize("bnd", [(11, 12), (22, 11)])
@pytest.mark.parametrize("q", [19, 27])
def test_duct_inflow_in_the_step(monkeypatch, q, bnd, storage):
    for n, dims in enumerate([(2, 2, 2), (5, 3, 2), (9, 2, 7), (33, 9, 30), (12, 65, 63), (10, 64, 64)]):
        monkeypatch.setenv("LBM_FAST_AXIS", str(0 if n > 3 else n % 3))
        print(f"D3Q{q} {storage} {bnd} {dims}", flush=True)
        shape = tuple(x + 2 for x in reversed(dims))
        rng = np.random.default_rng(n)
        mom = [1.0 + 0.01 * rng.random(shape)] + [0.03 * rng.random(shape) for _ in range(3)]
        got = []
        for fold in ("0", "1", None):
            if fold is None:
                monkeypatch.delenv("LBM_INFLOW_FOLD")
            else:
                monkeypatch.setenv("LBM_INFLOW_FOLD", fold)
            with Domain(q, dims, storage, iturb_pos=1, ibgk=3, ihrr=1, ivreman=1, smagorinsky=0.17, kinevisc=0.02, ibnd=1,
                        jbnd=bnd[0], kbnd=bnd[1]) as d:
                d.set_inflow(0.04, 20.0)
                d.init_equilibrium(*mom)
                d.step(0, 4)
                f = d.get_state()
                d.set_state(f)
                d.step(4, 3)
                got.append(d.get_state().tobytes())
        assert got[0] == got[1] == got[2]
