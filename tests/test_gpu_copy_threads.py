"""Records in and out of several contexts by several threads at once: large copies, which share the device's
page-locked slots and threads, beside ones that fit a slot.  Everything comes back as it went in."""
import threading

import numpy as np
import pytest

from lbm_amd.domain import Domain

pytestmark = pytest.mark.gpu


def test_contexts_of_several_threads():
    sizes = [(96, 48, 40), (12, 10, 8), (64, 64, 30), (20, 9, 7)]     # records of 16, 0.1, 10 and 0.2 MB
    wrong = []

    def work(n, dims):
        rng = np.random.default_rng(n)
        for rep in range(6):
            with Domain(19, dims, "f32", ibgk=2, kinevisc=0.1) as d:
                f = rng.random(d.shape_f, np.float32)
                for _ in range(3):
                    d.set_state(f)
                    if not np.array_equal(d.get_state(), f):
                        wrong.append((dims, rep))
        print(f"thread {n}: {dims} done", flush=True)

    threads = [threading.Thread(target=work, args=a) for a in enumerate(sizes)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not wrong
