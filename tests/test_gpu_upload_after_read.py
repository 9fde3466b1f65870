"""Setting a model after a field was read costs no more than before it, in a new
solver beside an earlier one's freed memory (19 ms for 8 where the read used the
stream of the uploads; the bar is 1.7, shortest of four)."""
import time

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _pair(make, slow):
    before, after = [], []
    for k in range(5):
        s = make()
        t0 = time.perf_counter()
        s.set_slowness(slow)
        t1 = time.perf_counter()
        s.solve()
        s.get_travel_time_field()
        t2 = time.perf_counter()
        s.set_slowness(slow)
        t3 = time.perf_counter()
        if k > 0:
            before.append(t1 - t0)
            after.append(t3 - t2)
        del s
    print("tuned %.2f ms, after a read %.2f ms"
          % (1e3 * min(before), 1e3 * min(after)), flush=True)
    return min(before), min(after)


def test_3d(ekx):
    dims, h = (257, 257, 193), 10.0
    slow = 1.0 / np.random.default_rng(1).uniform(2000.0, 5000.0,
                                                  256 * 256 * 192)

    def make():
        s = ekx.Solver3D()
        s.initialize(ekx.SolverOptions(number_of_sweeps=0),
                     ekx.Geometry3D(*dims, h))
        s.set_source((100.0, 100.0, 100.0))
        return s
    before, after = _pair(make, slow)
    assert after <= 1.7 * before


def test_2d(ekx):
    nx, nz = 4001, 1001
    slow = 1.0 / np.random.default_rng(2).uniform(2000.0, 5000.0,
                                                  (nx - 1) * (nz - 1))

    def make():
        s = ekx.Solver2D()
        s.initialize(ekx.SolverOptions(number_of_sweeps=0),
                     ekx.Geometry2D(nx, nz, 10.0))
        s.set_source((100.0, 100.0))
        return s
    before, after = _pair(make, slow)
    assert after <= 1.7 * before
