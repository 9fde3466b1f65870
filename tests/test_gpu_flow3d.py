"""Solves in one flow launch (the default for grids whose columns are all
resident) at the edges of their tiles, step groups and range: against the
oracle bit for bit in FP64, against the launches per diagonal (asked for by
naming a chunk depth) in the FP32 modes; batches, a grid with too many
columns, and solvers on several threads."""
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _inputs(nx, ny, nz, d, seed):
    rng = np.random.default_rng(seed)
    slow = 1.0 / rng.uniform(1800.0, 5200.0, (nx - 1) * (ny - 1) * (nz - 1))
    ext = [(n - 1) * h for n, h in zip((nx, ny, nz), d)]
    return slow, tuple(float(rng.uniform(0.0, e)) for e in ext), ext


def _solver(ekx, dims, d, slow, **options):
    s = ekx.Solver3D()
    s.initialize(ekx.SolverOptions(**options), ekx.Geometry3D(*dims, *d))
    s.set_slowness(slow)
    return s


@pytest.mark.parametrize("dims", [(3, 3, 3), (8, 8, 4), (9, 8, 5), (8, 16, 6),
                                  (17, 9, 7), (16, 25, 30), (41, 23, 64)])
@pytest.mark.parametrize("d", [(10.0, 10.0, 10.0), (10.0, 12.5, 8.0)])
@pytest.mark.parametrize("radius", [-1, 0, 4])
def test_edges(ekx, oracle, dims, d, radius):
    slow, src, ext = _inputs(*dims, d, sum(dims) + radius)
    print("case", dims, d, radius, flush=True)
    s = _solver(ekx, dims, d, slow, number_of_sweeps=2,
                factored_radius=radius)
    # an interior source, two opposite corners, the first one again
    for x in (src, (0.0, 0.0, 0.0), tuple(ext), src):
        s.set_source(x)
        s.solve()
        assert s.get_stats().kernel_launches == 1
        ref = oracle.solve3d(oracle.geometry3d(*dims, *d), slow, x, 2, radius)
        assert np.array_equal(s.get_travel_time_field(), ref), x


@pytest.mark.parametrize("precision", ["FP64", "FP32", "FP32_POLISH"])
@pytest.mark.parametrize("sweeps", [0, 1, 3])
def test_equals_the_diagonals(ekx, precision, sweeps):
    dims, d = (49, 39, 33), (10.0, 10.0, 10.0)
    slow, src, _ = _inputs(*dims, d, 7)
    print("case", precision, sweeps, flush=True)
    out = []
    for chunk in (0, 8):
        s = _solver(ekx, dims, d, slow, number_of_sweeps=sweeps,
                    factored_radius=3, chunk_planes=chunk,
                    precision=getattr(ekx.Precision, precision))
        s.set_source(src)
        s.solve()
        out.append((s.get_travel_time_field(), s.get_stats()))
    assert np.array_equal(out[0][0], out[1][0])
    flow, diagonals = out[0][1], out[1][1]
    assert flow.kernel_launches <= 2 < diagonals.kernel_launches
    for name in ("updates", "updates_fp64", "iterations_run", "tiled"):
        assert getattr(flow, name) == getattr(diagonals, name)


@pytest.mark.parametrize("precision", ["FP64", "FP32"])
@pytest.mark.parametrize("dims", [(64, 32, 9), (72, 32, 9), (130, 70, 9),
                                  (70, 261, 12)])
def test_runs_of_columns(ekx, dims, precision):
    """One XCD just full (32 columns), one column more, and runs that end
    within a row of columns on several XCDs."""
    slow, src, _ = _inputs(*dims, (10.0,) * 3, 5)
    print("case", dims, precision, flush=True)
    out = []
    for chunk in (0, 8):
        s = _solver(ekx, dims, (10.0,) * 3, slow, number_of_sweeps=2,
                    factored_radius=2, chunk_planes=chunk,
                    precision=getattr(ekx.Precision, precision))
        s.set_source(src)
        s.solve()
        assert (s.get_stats().kernel_launches == 1) == (chunk == 0)
        out.append(s.get_travel_time_field())
    assert np.array_equal(*out)


@pytest.mark.parametrize("precision", ["FP64", "FP32_POLISH"])
@pytest.mark.parametrize("shared", [False, True])
def test_batch_beyond_the_device(ekx, precision, shared):
    """More columns than the device holds: problems follow each other through
    it, each as the diagonals solve it."""
    rng = np.random.default_rng(3)
    d, problems = (10.0,) * 3, []
    slow = None
    for k in range(66):
        dims = (64, 49, 6) if shared else \
            tuple(int(v) for v in (*rng.integers(40, 73, 2),
                                   rng.integers(4, 12)))
        new, src, _ = _inputs(*dims, d, k)
        slow = new if not shared or slow is None else slow
        problems.append((ekx.Geometry3D(*dims, *d), slow, src))
    columns = sum(((g.nx + 7) // 8) * ((g.ny + 7) // 8)
                  for g, _, _ in problems)
    assert columns > 2048
    print("case", precision, shared, columns, flush=True)
    out = []
    for chunk in (0, 8):
        b = ekx.Batch3D()
        b.initialize(ekx.SolverOptions(
            number_of_sweeps=1, factored_radius=2, chunk_planes=chunk,
            precision=getattr(ekx.Precision, precision)), problems)
        for _ in range(2):
            b.solve()
        assert (b.get_stats().kernel_launches <= 2) == (chunk == 0)
        out.append([b.get_travel_time_field(k) for k in range(len(problems))])
    assert all(np.array_equal(x, y) for x, y in zip(*out))


def test_batch_of_uneven_grids(ekx, oracle):
    rng = np.random.default_rng(11)
    problems, refs = [], []
    for k in range(6):
        dims = tuple(int(v) for v in rng.integers(5, 40, 3))
        slow, src, _ = _inputs(*dims, (10.0,) * 3, k)
        problems.append((ekx.Geometry3D(*dims, 10.0), slow, src))
        refs.append(oracle.solve3d(oracle.geometry3d(*dims, 10.0), slow, src,
                                   1, 2))
    b = ekx.Batch3D()
    b.initialize(ekx.SolverOptions(number_of_sweeps=1, factored_radius=2),
                 problems)
    b.solve()
    assert b.get_stats().kernel_launches == 1
    for k, ref in enumerate(refs):
        assert np.array_equal(b.get_travel_time_field(k), ref), k


def test_more_columns_than_the_device_holds(ekx, oracle):
    dims, d = (801, 801, 3), (10.0,) * 3
    slow, src, _ = _inputs(*dims, d, 3)
    s = _solver(ekx, dims, d, slow, number_of_sweeps=1, factored_radius=2)
    s.set_source(src)
    s.solve()
    assert s.get_stats().kernel_launches > 1
    ref = oracle.solve3d(oracle.geometry3d(*dims, *d), slow, src, 1, 2)
    assert np.array_equal(s.get_travel_time_field(), ref)


def test_several_threads(ekx, oracle):
    """Four solvers at once, together with more columns than the device
    holds: whichever route each takes, the field is the oracle's."""
    dims, d = (217, 217, 12), (10.0,) * 3
    slow, _, _ = _inputs(*dims, d, 21)
    sources = [(310.0, 420.0, 55.0), (1900.0, 77.0, 11.0),
               (1000.0, 2000.0, 90.0), (5.0, 1200.0, 100.0)]
    refs = [oracle.solve3d(oracle.geometry3d(*dims, *d), slow, x, 1, 2)
            for x in sources]
    same = [False] * len(sources)

    def work(k):
        s = _solver(ekx, dims, d, slow, number_of_sweeps=1,
                    factored_radius=2)
        s.set_source(sources[k])
        good = True
        for _ in range(3):
            s.solve()
            good = good and np.array_equal(s.get_travel_time_field(), refs[k])
        same[k] = good

    threads = [threading.Thread(target=work, args=(k,))
               for k in range(len(sources))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert all(same), same
