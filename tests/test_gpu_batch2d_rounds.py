"""Large 2D batches take their rounds of one workgroup a CU one after the other:
eight rounds take no longer than eight times one (two workgroups on a CU spill
the Infinity Cache: 8.7 times; the bar is 8.4, shortest of ten), and each field
is a single solve's, in batches of few and of many problems."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _batch(ekx, g, slow, n, seed):
    rng = np.random.default_rng(seed)
    sources = [(float(rng.uniform(0, (g.nx - 1) * 10.0)),
                float(rng.uniform(0, (g.nz - 1) * 10.0))) for _ in range(n)]
    b = ekx.Batch2D()
    o = ekx.SolverOptions(number_of_sweeps=2, factored_radius=3)
    b.initialize(o, [(g, slow, x) for x in sources])
    times = []
    for _ in range(10):
        b.solve()
        times.append(b.get_stats().last_solve_ms)
    for i in (0, n // 2, n - 1):
        s = ekx.Solver2D()
        s.initialize(o, g)
        s.set_slowness(slow)
        s.set_source(sources[i])
        s.solve()
        assert np.array_equal(b.get_travel_time_field(i),
                              s.get_travel_time_field()), i
    return min(times)


def test_eight_rounds(ekx):
    g = ekx.Geometry2D(201, 201, 10.0)
    rng = np.random.default_rng(2)
    slow = 1.0 / rng.uniform(2000.0, 5000.0, 200 * 200)
    one, eight = _batch(ekx, g, slow, 256, 3), _batch(ekx, g, slow, 2048, 4)
    print("tuned 256: %.2f ms, 2048: %.2f ms" % (one, eight), flush=True)
    assert eight <= 8.4 * one


@pytest.mark.parametrize("nx,nz", [(40, 64), (33, 65), (17, 129), (21, 257),
                                   (9, 530), (6, 1000)])
def test_many_problems(ekx, nx, nz):
    g = ekx.Geometry2D(nx, nz, 10.0)
    rng = np.random.default_rng(nx)
    slow = 1.0 / rng.uniform(2000.0, 5000.0, (nx - 1) * (nz - 1))
    print("case", nx, nz, flush=True)
    _batch(ekx, g, slow, 700, nz)
