"""Ducts on both sides of the sizes from which the step kernel writes their inflow/outflow planes by default, for each
storage: the same state, bit for bit, as with the planes in a launch of their own and in the step."""
import numpy as np
import pytest

from lbm_amd.domain import Domain

pytestmark = pytest.mark.gpu

DUCTS = {"f32": [(20, 63, 65), (20, 64, 64)], "f16s": [(64, 120, 119), (64, 120, 120), (65, 64, 64), (65, 241, 17)],
         "bf16s": [(64, 144, 100), (65, 17, 241)], "f64": [(160, 64, 64), (160, 17, 241), (161, 241, 17)]}


@pytest.mark.parametrize("q", [19, 27])
@pytest.mark.parametrize("storage", DUCTS)
def test_defaults_of_ducts(monkeypatch, storage, q):
    for dims in DUCTS[storage]:
        print(f"D3Q{q} {storage} {dims}", flush=True)
        shape = tuple(x + 2 for x in reversed(dims))
        rng = np.random.default_rng(5)
        mom = [1.0 + 0.01 * rng.random(shape)] + [0.03 * rng.random(shape) for _ in range(3)]
        got = []
        for fold in ("0", "1", None):
            if fold is None:
                monkeypatch.delenv("LBM_INFLOW_FOLD")
            else:
                monkeypatch.setenv("LBM_INFLOW_FOLD", fold)
            with Domain(q, dims, storage, iturb_pos=1, ibgk=3, ihrr=1, ivreman=1, smagorinsky=0.17, kinevisc=0.02, ibnd=1,
                        jbnd=11, kbnd=12) as d:
                d.set_inflow(0.04, 20.0)
                d.init_equilibrium(*mom)
                d.step(0, 3)
                got.append(d.get_state().tobytes())
        assert got[0] == got[1] == got[2]
