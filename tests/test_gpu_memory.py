"""Device memory that a context holds, against what its inputs and its size account for.

hipMemGetInfo counts whole allocations, each rounded up to 2 MiB at most; a context has fewer than 16 of
them, hence the 32 MiB of slack, which is far below what each test looks for.
"""
import numpy as np
import pytest
import torch

from lbm_amd.domain import Domain

pytestmark = pytest.mark.gpu

SLACK = 32 << 20


def free_bytes():
    torch.cuda.synchronize()
    return torch.cuda.mem_get_info()[0]


def test_averaging_sums_are_freed():
    dims = (128, 96, 64)
    sums = 6 * np.prod([n + 2 for n in dims]) * 8
    held = []
    for n in range(4):
        with Domain(19, dims, "f64", ibgk=2, kinevisc=0.1) as d:
            d.set_averaging()
            print(f"context {n}: {d.info()}", flush=True)
        held.append(free_bytes())
    # from the second context on nothing is set up any more; each lost sums would take 40 MB
    assert sums > SLACK and held[0] - held[-1] < SLACK


def test_window_scratch_is_given_back():
    """A window whose scratch and fields outgrow a record of the state: what stays is what the context needs
    afterwards (populations, the three fields, at most a record's staging memory)."""
    dims, n, window = (16, 128, 128), 200, 201 * 128 * 128 * 4
    record = 19 * np.prod([x + 2 for x in dims]) * 4
    before = free_bytes()
    with Domain(19, dims, "f32", ibgk=2, kinevisc=0.1, ibnd=1, kbnd=12) as d:
        for seed in (1, 2):
            d.generate_turbulence(n, 1e-3, seed, return_fields=False)
            held = before - free_bytes()
            print(f"seed {seed}: {held >> 20} MB held", flush=True)
            # scratch (4 variables of 201 x 65 x 256 complex values) and fields took 267 MB more
            assert held < d.info()["device_bytes"] + 3 * window + record + SLACK


def test_adjoint_holds_its_workspace_only():
    """The force gradient needs its FP64 accumulator (three per-cell arrays) beside what a run without it holds, also
    where the context's staging memory is no larger than an FP32 start's."""
    dims = (160, 128, 96)
    cells = np.prod([n + 2 for n in dims])
    with Domain(19, dims, "f32", ibgk=2, kinevisc=0.1) as d:
        m = [np.full(d.shape_cell, v, np.float32) for v in (1.0, 0.01, 0.0, 0.0)]
        assert d.lib.lbm_init_equilibrium(d.h, *[a.ctypes.data for a in m], 4, 0) == 0
        d.set_external_forcing(np.full(d.shape_cell + (3,), 1e-6, np.float32))
        d.step(0, 1)
        box = ((2, 9),) * 3
        d.adjoint(1, 2, 2, box, grad_force=False)
        before = free_bytes()
        d.adjoint(3, 2, 2, box, grad_force=True)
        more = before - free_bytes()
        accumulator = 3 * d.info()["plane"] * 8
        print(f"{more >> 20} MB more, accumulator {accumulator >> 20} MB", flush=True)
        # staging memory of 24 bytes a cell in the place of 16 would be 17 MB more still; allocations end at 2 MiB
        assert 8 * cells > 16e6 and more < accumulator + (8 << 20)
