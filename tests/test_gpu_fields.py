"""Per-cell values in and out of the device order (fields.h): records, moments, averages and forcing
fields whose extents end inside, at and just past a tile (64 x 4 cells along i, j with i contiguous;
8 cells along i x 32 along the contiguous axis otherwise), for each contiguous axis.

A record read back right after it was set is the same bit for bit, ghosts included (FP32 and FP64
storage of values of that kind).  Moments are sums of at most 27 populations below 0.35 and a
quotient by a density of about 1: within 27 * 2^-24 (FP32) or 27 * 2^-53 (FP64) times 2 of the FP64
sums.  A forced run does the same arithmetic for each contiguous axis: 4 steps within 4 * 8 units in
the last place of a population below 0.5, 32 * 2^-25 = 1e-6 (FP32), 1.8e-15, taken as 4e-15 (FP64).
"""
import numpy as np
import pytest

from lbm_amd.domain import Domain, LBMError
from lbm_amd.lattice import lattice

pytestmark = pytest.mark.gpu

DIMS = [(2, 2, 2), (6, 30, 31), (7, 31, 30), (62, 9, 4), (63, 33, 5), (13, 6, 62)]


def record(q, dims, dt, seed):
    nx, ny, nz = dims
    rng = np.random.default_rng(seed)
    w = lattice(q).w
    return (w * (1.0 + 0.05 * rng.uniform(-1, 1, (nz + 2, ny + 2, nx + 2, q)))).astype(dt)


@pytest.mark.parametrize("axis", [0, 1, 2])
@pytest.mark.parametrize("dims", DIMS)
@pytest.mark.parametrize("q,storage", [(27, "f32"), (19, "f64")])
def test_records_moments_and_forcing(monkeypatch, axis, dims, q, storage):
    dt = np.float64 if storage == "f64" else np.float32
    eps = np.finfo(dt).eps
    print(f"D3Q{q} {storage} {dims}, contiguous axis {axis}", flush=True)
    f0 = record(q, dims, dt, sum(dims))
    F = (1e-4 * np.random.default_rng(1).standard_normal(f0.shape[:3] + (3,)))
    theta = 300.0 + np.random.default_rng(2).uniform(-2, 2, f0.shape[:3])
    out = []
    for ax in (axis, 0):
        monkeypatch.setenv("LBM_FAST_AXIS", str(ax))
        with Domain(q, dims, storage, ibgk=2, kinevisc=0.1, ibnd=0, jbnd=0, kbnd=0) as d:
            d.set_state(f0)
            assert np.array_equal(d.get_state(), f0)
            lat = lattice(q)
            f = f0.astype(np.float64)
            rho = f.sum(-1)
            want = [rho] + [(f * c).sum(-1) / rho for c in (lat.cx, lat.cy, lat.cz)]
            for got, ref in zip(d.macrovars(), want):
                assert got.dtype == dt and np.abs(got - ref).max() < 27 * eps
            d.set_external_forcing(F)
            d.set_buoyancy(theta, 300.0, 1e-4)
            d.step(0, 4)
            out.append(d.get_state().astype(np.float64))
            d.set_averaging(True)
            d.step(4, 1)
            m = d.macrovars(np.float64)
            inner = (slice(1, -1),) * 3
            a = d.averages(np.float64)
            for got, ref in zip(a[:3], m[1:]):
                assert np.abs(got[inner] - ref[inner]).max() < 27 * eps
                got[inner] = 0.0
                assert not got.any()           # ghosts hold zeros
    assert np.abs(out[0] - out[1]).max() < (4e-15 if storage == "f64" else 1e-6)


@pytest.mark.parametrize("axis", [0, 1, 2])
@pytest.mark.parametrize("cell", [(0, 0, 0), (1, 9, 5), (8, 8, 4), (4, 33, 6)])
def test_one_bad_cell_is_seen(monkeypatch, axis, cell):
    """A single negative density anywhere in the padded grid makes the moments unstable."""
    dims = (7, 32, 5)
    monkeypatch.setenv("LBM_FAST_AXIS", str(axis))
    f0 = record(19, dims, np.float32, 5)
    f0[cell[2], cell[1], cell[0]] *= -1.0
    with Domain(19, dims, "f32", ibgk=2, kinevisc=0.1, ibnd=11, jbnd=11, kbnd=11) as d:
        d.set_state(f0)
        with pytest.raises(LBMError, match="0 non-finite moments, 1 cells with density <= 0"):
            d.macrovars()
