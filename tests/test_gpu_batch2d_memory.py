"""The working memory of a large 2D batch is bounded: its problems share it slice
by slice, and each field is the single solve's, at the ends of the slices
too."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _free_bytes():
    hip = ctypes.CDLL("libamdhip64.so.7", mode=ctypes.RTLD_GLOBAL)
    free, total = ctypes.c_size_t(), ctypes.c_size_t()
    assert hip.hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0
    return free.value


def test_slices(ekx):
    """4096 problems of 201 x 201: fields 1.32 GB, skewed times of all 6.8 GB,
    of a slice at most 4.3 GB."""
    n = 4096
    g = ekx.Geometry2D(201, 201, 10.0)
    rng = np.random.default_rng(9)
    slow = 1.0 / rng.uniform(2000.0, 5000.0, 200 * 200)
    sources = [(float(rng.uniform(0, 2000.0)), float(rng.uniform(0, 2000.0)))
               for _ in range(n)]
    o = ekx.SolverOptions(number_of_sweeps=1, factored_radius=3)
    small = ekx.Batch2D()           # (the library's own first allocations)
    small.initialize(o, [(g, slow, sources[0])])
    small.solve()
    before = _free_bytes()
    b = ekx.Batch2D()
    b.initialize(o, [(g, slow, x) for x in sources])
    used = before - _free_bytes()
    print("tuned %.2f GB" % (used * 1e-9), flush=True)
    for _ in range(2):
        b.solve()
    assert b.get_stats().kernel_launches == 2
    for i in (0, 1, 2046, 2047, 2048, 2049, 4094, 4095):
        s = ekx.Solver2D()
        s.initialize(o, g)
        s.set_slowness(slow)
        s.set_source(sources[i])
        s.solve()
        assert np.array_equal(b.get_travel_time_field(i),
                              s.get_travel_time_field()), i
    assert used < 6.0e9


def test_uneven_slices(ekx):
    """Grids of one band and of sixteen, one too tall for bands, and models out
    of range, over several slices (9.4 GB of skewed times in all)."""
    rng = np.random.default_rng(10)
    o = ekx.SolverOptions(number_of_sweeps=1, factored_radius=2)
    problems = []
    for i in range(800):
        nx, nz = [(1500, 1000), (300, 64), (60, 1030), (1000, 900)][i % 4]
        scale = 2.0 ** -360 if i % 7 == 3 else 1.0
        if i < 8:
            slow = scale / rng.uniform(2000.0, 5000.0, (nx - 1) * (nz - 1))
        else:
            slow = problems[i % 4][1]
        problems.append((ekx.Geometry2D(nx, nz, 10.0), slow,
                         (float(rng.uniform(0, (nx - 1) * 10.0)),
                          float(rng.uniform(0, (nz - 1) * 10.0)))))
    b = ekx.Batch2D()
    b.initialize(o, problems)
    b.solve()
    print("launches", b.get_stats().kernel_launches, flush=True)
    assert b.get_stats().kernel_launches > 3
    for i in [*range(8), *range(260, 272), *range(528, 540), 798, 799]:
        s = ekx.Solver2D()
        s.initialize(o, problems[i][0])
        s.set_slowness(problems[i][1])
        s.set_source(problems[i][2])
        s.solve()
        assert np.array_equal(b.get_travel_time_field(i),
                              s.get_travel_time_field()), i
