"""Waits of the one-launch solves: their bound follows the number of sweeps
where problems wait for others to finish, and past the bound the solve, and
those after it, go by diagonals."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def test_a_problem_waits_for_another_to_finish(ekx):
    """Two problems of 2025 columns each on 2048 resident waves: the second
    starts when the first has done its 1048 sweeps, some hundreds of ms
    later.  Each field is that of its own solve."""
    dims, h, sweeps = (360, 360, 4), 10.0, 130
    rng = np.random.default_rng(8)
    slow = 1.0 / rng.uniform(1800.0, 5200.0, 359 * 359 * 3)
    g = ekx.Geometry3D(*dims, h)
    sources = [(100.0, 3300.0, 12.0), (2000.0, 1500.0, 25.0)]
    o = ekx.SolverOptions(number_of_sweeps=sweeps, factored_radius=2)
    b = ekx.Batch3D()
    b.initialize(o, [(g, slow, x) for x in sources])
    b.solve()
    st = b.get_stats()
    print("batch", st.last_solve_ms, "ms", flush=True)
    assert st.kernel_launches == 1
    for k, x in enumerate(sources):
        s = ekx.Solver3D()
        s.initialize(o, g)
        s.set_slowness(slow)
        s.set_source(x)
        s.solve()
        assert s.get_stats().kernel_launches == 1
        assert np.array_equal(s.get_travel_time_field(),
                              b.get_travel_time_field(k)), k


@pytest.mark.parametrize("precision", ["FP64", "FP32_POLISH"])
@pytest.mark.parametrize("batch", [False, True])
def test_past_the_bound_by_diagonals(ekx, oracle, precision, batch):
    """A bound that no wait meets: every wave gives up and ends, and the
    field is the diagonals'."""
    dims, h = (129, 73, 21), 10.0
    rng = np.random.default_rng(12)
    slow = 1.0 / rng.uniform(1800.0, 5200.0, 128 * 72 * 20)
    g = ekx.Geometry3D(*dims, h)
    src = (700.0, 310.0, 95.0)
    print("case", precision, batch, flush=True)

    def make(chunk):
        o = ekx.SolverOptions(number_of_sweeps=2, factored_radius=2,
                              chunk_planes=chunk,
                              precision=getattr(ekx.Precision, precision))
        s = ekx.Batch3D() if batch else ekx.Solver3D()
        if batch:
            s.initialize(o, [(g, slow, src)] * 2)
            return s, lambda: s.get_travel_time_field(1)
        s.initialize(o, g)
        s.set_slowness(slow)
        s.set_source(src)
        return s, s.get_travel_time_field

    by_diagonals, field = make(8)
    by_diagonals.solve()
    ref = field()
    if precision == "FP64":
        assert np.array_equal(ref, oracle.solve3d(
            oracle.geometry3d(*dims, h), slow, src, 2, 2))
    one = 1 if precision == "FP64" else 2
    s, field = make(0)
    s.set_wait_bound(0.0)
    s.solve()
    assert s.get_stats().kernel_launches > one
    assert np.array_equal(field(), ref)
    # the device stays shared: no second try
    s.set_wait_bound(-1.0)
    s.solve()
    assert s.get_stats().kernel_launches > one
    assert np.array_equal(field(), ref)
    # a new setup tries again
    s, field = make(0)
    s.solve()
    assert s.get_stats().kernel_launches == one
    assert np.array_equal(field(), ref)
    with pytest.raises(ValueError):
        s.set_wait_bound(1e10)


def test_threads_take_turns(ekx, oracle):
    """Three solvers of 1089 columns on three threads: the device holds one at a
    time, and the others wait for their turn instead of going by diagonals."""
    import threading
    dims, h = (257, 257, 40), 10.0
    rng = np.random.default_rng(14)
    slow = 1.0 / rng.uniform(1800.0, 5200.0, 256 * 256 * 39)
    sources = [(310.0, 420.0, 55.0), (1900.0, 77.0, 11.0),
               (1000.0, 2000.0, 90.0)]
    launches, same = [[] for _ in sources], [False] * len(sources)
    solvers = []
    for x in sources:
        s = ekx.Solver3D()
        s.initialize(ekx.SolverOptions(number_of_sweeps=2, factored_radius=2),
                     ekx.Geometry3D(*dims, h))
        s.set_slowness(slow)
        s.set_source(x)
        s.solve()
        solvers.append(s)
    refs = [oracle.solve3d(oracle.geometry3d(*dims, h), slow, x, 2, 2)
            for x in sources]

    def work(k):
        for _ in range(6):
            solvers[k].solve()
            launches[k].append(solvers[k].get_stats().kernel_launches)
        same[k] = np.array_equal(solvers[k].get_travel_time_field(), refs[k])
    threads = [threading.Thread(target=work, args=(k,))
               for k in range(len(sources))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    print("launches", launches, flush=True)
    assert all(same), same
    assert launches == [[1] * 6] * 3
