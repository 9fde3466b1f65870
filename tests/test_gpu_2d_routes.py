"""The routes of 2D solves: bands with and without range tests of their roots
and levels, alone and side by side in one batch; each problem by its own
route, whatever the others take.  Every field is the single solve's, which is
the oracle's (the 1e-12 bar of the 2D solver: hypot's ulp in the box)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

TINY, HUGE = 2.0 ** -360, 1e9             # times a slowness: out of range


def _single(ekx, g, slow, src, sweeps=1, radius=3):
    s = ekx.Solver2D()
    s.initialize(ekx.SolverOptions(number_of_sweeps=sweeps,
                                   factored_radius=radius), g)
    s.set_slowness(slow)
    s.set_source(src)
    return s


def _check(got, ref, floor):
    rel = np.abs(got - ref) / np.maximum(ref, floor)
    assert rel.max() <= 1e-12, rel.max()


@pytest.mark.parametrize("nx,nz", [(9, 12), (8, 65), (30, 200), (11, 530),
                                   (13, 769), (7, 1024), (9, 1030)])
@pytest.mark.parametrize("dz", [10.0, 12.5])
@pytest.mark.parametrize("scale", [TINY, HUGE])
def test_out_of_range_alone(ekx, oracle, nx, nz, dz, scale):
    rng = np.random.default_rng(nx + nz)
    slow = scale / rng.uniform(1500.0, 5500.0, (nx - 1) * (nz - 1))
    src = (0.4 * (nx - 1) * 10.0, 0.7 * (nz - 1) * dz)
    print("case", nx, nz, dz, scale, flush=True)
    for radius, sweeps in ((3, 1), (-1, 2)):
        s = _single(ekx, ekx.Geometry2D(nx, nz, 10.0, dz), slow, src, sweeps,
                    radius)
        for _ in range(2):
            s.solve()
            _check(s.get_travel_time_field(),
                   oracle.solve2d(oracle.geometry2d(nx, nz, 10.0, dz), slow,
                                  src, sweeps, radius), slow.min() * 10.0)


@pytest.mark.parametrize("dims", [
    [(20, 30, 1.0), (20, 30, TINY), (40, 700, 1.0), (15, 1000, HUGE)],
    [(20, 30, 1.0), (9, 1100, 1.0), (12, 100, TINY), (9, 1100, TINY)],
    [(9, 1100, 1.0), (6, 1300, 1.0)],
    [(70, 50, TINY), (50, 200, TINY), (12, 10, TINY)],
    [(30, 40, 1.0), (30, 550, 1.0), (30, 1024, 1.0), (30, 64, 1.0)]])
def test_side_by_side(ekx, dims):
    rng = np.random.default_rng(len(dims))
    problems = []
    for nx, nz, scale in dims * 3:
        slow = scale / rng.uniform(1500.0, 5500.0, (nx - 1) * (nz - 1))
        problems.append((ekx.Geometry2D(nx, nz, 10.0), slow,
                         (float(rng.uniform(0, (nx - 1) * 10.0)),
                          float(rng.uniform(0, (nz - 1) * 10.0)))))
    print("case", dims, flush=True)
    b = ekx.Batch2D()
    b.initialize(ekx.SolverOptions(number_of_sweeps=1, factored_radius=3),
                 problems)
    for _ in range(2):
        b.solve()
    for i, problem in enumerate(problems):
        s = _single(ekx, *problem)
        s.solve()
        assert np.array_equal(b.get_travel_time_field(i),
                              s.get_travel_time_field()), i


def test_out_of_range_is_no_slower_than_half(ekx):
    """The same steps with range tests: 201 x 201 took 2.6 times as long by
    levels; the bar is 2 (about 1.3 expected), shortest of ten."""
    rng = np.random.default_rng(1)
    slow = 1.0 / rng.uniform(1500.0, 5500.0, 200 * 200)
    times = []
    for scale in (1.0, TINY):
        s = _single(ekx, ekx.Geometry2D(201, 201, 10.0), scale * slow,
                    (371.0, 402.0), 2)
        ms = []
        for _ in range(10):
            s.solve()
            ms.append(s.get_stats().last_solve_ms)
        times.append(min(ms))
    print("tuned", times, flush=True)
    assert times[1] <= 2.0 * times[0]
