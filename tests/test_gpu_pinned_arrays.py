"""Records, moments, averages and forcing from and to arrays that the caller has page-locked (all of them, or some of
a call's): the same bytes as with ordinary ones, for copies of one slot and of many."""
import ctypes as C

import numpy as np
import pytest

from lbm_amd.domain import Domain, load_library

pytestmark = pytest.mark.gpu


class Pinned:
    """numpy arrays in page-locked memory of the runtime that the library runs on."""

    def __init__(self):
        load_library()
        self.hip = C.CDLL("libamdhip64.so.7")
        self.held = []

    def empty(self, shape, dtype):
        n = int(np.prod(shape)) * np.dtype(dtype).itemsize
        p = C.c_void_p()
        assert self.hip.hipHostMalloc(C.byref(p), C.c_size_t(n), C.c_uint(0)) == 0
        self.held.append(p)
        return np.frombuffer((C.c_char * n).from_address(p.value), dtype).reshape(shape)

    def free(self):
        for p in self.held:
            self.hip.hipHostFree(p)


@pytest.mark.parametrize("dims", [(14, 9, 8), (90, 62, 40)])
def test_page_locked_arrays(dims):
    ptr = lambda a: a.ctypes.data_as(C.c_void_p)
    mem = Pinned()
    with Domain(19, dims, "f32", ibgk=2, kinevisc=0.1) as d:
        rng = np.random.default_rng(1)
        f = mem.empty(d.shape_f, np.float32)
        f[...] = 1.0 / 19 + 1e-3 * rng.random(d.shape_f, np.float32)
        print(f"D3Q19 {dims}, record of {f.nbytes} bytes", flush=True)
        d.set_state(f)
        back = mem.empty(d.shape_f, np.float32)
        assert d.lib.lbm_get_state(d.h, ptr(back), 4) == 0
        assert np.array_equal(back, f) and np.array_equal(d.get_state(), f)
        F = mem.empty(d.shape_cell + (3,), np.float32)
        F[...] = 1e-6
        d.set_external_forcing(F)
        d.set_averaging()
        d.step(1, 3)
        want = d.macrovars()
        for pinned in (15, 5, 8):
            got = [(mem.empty if pinned >> q & 1 else np.empty)(d.shape_cell, np.float32) for q in range(4)]
            assert d.lib.lbm_get_macros(d.h, *[ptr(a) for a in got], 4) == 0
            assert all(np.array_equal(a, b) for a, b in zip(got, want))
        want = d.averages()
        got = [mem.empty(d.shape_cell, np.float32), None, np.empty(d.shape_cell, np.float32), None]
        n = C.c_int()
        assert d.lib.lbm_get_averages(d.h, *[ptr(a) if a is not None else None for a in got], C.byref(n), 4) == 0
        assert n.value == 3 and np.array_equal(got[0], want[0]) and np.array_equal(got[2], want[2])
    mem.free()
