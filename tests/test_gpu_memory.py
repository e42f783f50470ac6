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
