"""Rows of n cells against rows of 2 n that hold the same field twice along a periodic contiguous axis: every
cell does the same arithmetic on the same values, so both halves are the short rows' bit for bit, wherever a
row ends (within 64 bytes, at them, where the padding that the step stores reaches the next row's unread
ghost).  Single domains and, over the same lengths, ensembles against lbm_step, for each storage.
"""
import numpy as np
import pytest

from lbm_amd import inputs
from lbm_amd.domain import Domain, Ensemble

pytestmark = pytest.mark.gpu

LENGTHS = (7, 8, 9, 16, 17, 31, 32, 33, 62, 63)
STORAGES = ["f32", "f64", "f16s", "bf16s"]
PHYS = dict(ibgk=3, ihrr=1, ivreman=1, smagorinsky=0.17, kinevisc=0.01, ibnd=1, jbnd=0, kbnd=12)


def domain(q, storage, n, copies=1, seed=None):
    """Inflow along i, closed k, j periodic and contiguous, with `copies` of one field of n cells along j."""
    nx, nz = 14, 6
    dt = np.float64 if storage == "f64" else np.float32
    f = inputs.perturbed_uniform_flow(q, (nx, n, nz), seed=n if seed is None else seed, u0=(0.05, 0, 0), order=3, dtype=dt)
    inner = np.concatenate([f[:, 1:-1]] * copies, 1)
    f = np.concatenate([inner[:, -1:], inner, inner[:, :1]], 1)
    turb = [np.concatenate([t] * copies, 2) for t in inputs.turbulence_fields(3, n, nz, 5, dtype=dt)[:3]]
    mask = np.zeros((nz + 2, n * copies + 2, nx + 2), np.uint8)
    for c in range(copies):
        mask[1:4, c * n + 2:c * n + 1 + max(2, n // 3), 4:7] = 1
    d = Domain(q, (nx, n * copies, nz), storage, **PHYS)
    d.set_state(f)
    d.set_inflow(0.05, 10.0)
    d.set_blanking(mask)
    d.set_turbulence(*turb, 5, 1e-3)
    return d


@pytest.mark.parametrize("q", [19, 27])
@pytest.mark.parametrize("storage", STORAGES)
def test_doubled_rows_are_bit_identical(storage, q):
    for n in LENGTHS:
        print(f"D3Q{q} {storage} rows of {n}", flush=True)
        out = []
        for copies in (1, 2):
            with domain(q, storage, n, copies) as d:
                d.step(1, 9)
                out.append(d.get_state())
        one, two = out
        assert np.isfinite(one).all()
        assert np.array_equal(two[:, 1:n + 1], one[:, 1:-1]) and np.array_equal(two[:, n + 1:-1], one[:, 1:-1])


@pytest.mark.parametrize("launch", [(256, 0), (64, 2)])
@pytest.mark.parametrize("storage", STORAGES)
def test_ensemble_rows_are_those_of_single_domains(storage, launch):
    print(f"{storage} ensemble of rows {LENGTHS}, launch {launch}", flush=True)
    a, b = ([domain(19, storage, n) for n in LENGTHS] for _ in range(2))
    ens = Ensemble(a)
    ens.set_launch(*launch)
    ens.step(1, 9)
    ens.synchronize()
    ens.close()
    for n, x, y in zip(LENGTHS, a, b):
        y.step(1, 9)
        assert np.array_equal(x.get_state(), y.get_state()), f"rows of {n}"
        x.close()
        y.close()
