"""The autotuner keeps what it has timed: the default shape as the default runs
it (the factored box inside chunks of 64 to 79 planes, FP64), the solve in
one launch where that is faster, and the tuned diagonals where it gives up."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _inputs(dims, seed, h=10.0):
    rng = np.random.default_rng(seed)
    cells = (dims[0] - 1) * (dims[1] - 1) * (dims[2] - 1)
    return rng, 1.0 / rng.uniform(1800.0, 5200.0, cells)


def test_default_shape_is_the_one_timed(ekx):
    """1800 problems of 65 x 65 x 70 run by whole columns of 70 planes with the
    box in the bulk launches: the tuned solves are no slower than the default
    (with the box timed in launches of its own the tuner took another depth,
    14% slower; the bar is 8%, shortest of four)."""
    dims, h, n = (65, 65, 70), 10.0, 1800
    rng, slow = _inputs(dims, 3)
    g = ekx.Geometry3D(*dims, h)
    b = ekx.Batch3D()
    b.initialize(ekx.SolverOptions(
        number_of_sweeps=1, factored_radius=2,
        launch_order=ekx.LaunchOrder.DIAGONALS),
        [(g, slow, tuple(float(rng.uniform(0, (m - 1) * h)) for m in dims))
         for _ in range(n)])

    def solve_ms():
        times = []
        for _ in range(4):
            b.solve()
            times.append(b.get_stats().last_solve_ms)
        return min(times), b.get_stats()
    before, default = solve_ms()
    fields = [b.get_travel_time_field(i) for i in (0, 899, 1799)]
    assert default.chunk_planes == 70
    chunk, chains = b.autotune()
    after, st = solve_ms()
    print("tuned", chunk, chains, before, after, flush=True)
    assert (st.chunk_planes, st.chains) == (chunk, chains)
    if chunk == default.chunk_planes:
        assert st.updates_factored == default.updates_factored
    for i, f in zip((0, 899, 1799), fields):
        assert np.array_equal(b.get_travel_time_field(i), f), i
    assert after <= 1.08 * before


@pytest.mark.parametrize("precision", ["FP64", "FP32_POLISH"])
@pytest.mark.parametrize("gives_up", [False, True])
def test_one_launch_is_a_candidate(ekx, precision, gives_up):
    dims, h = (129, 121, 40), 10.0
    _, slow = _inputs(dims, 4)
    s = ekx.Solver3D()
    s.initialize(ekx.SolverOptions(
        number_of_sweeps=2, factored_radius=2,
        precision=getattr(ekx.Precision, precision)),
        ekx.Geometry3D(*dims, h))
    s.set_slowness(slow)
    s.set_source((640.0, 310.0, 77.0))
    s.solve()
    ref = s.get_travel_time_field()
    one = 1 if precision == "FP64" else 2
    assert s.get_stats().kernel_launches == one
    print("case", precision, gives_up, flush=True)
    if gives_up:
        s.set_wait_bound(0.0)
    chunk, chains = s.autotune()
    s.set_wait_bound(-1.0)
    s.solve()
    st = s.get_stats()
    assert (st.kernel_launches > one) == gives_up
    assert (st.chunk_planes, st.chains) == (chunk, chains)
    assert np.array_equal(s.get_travel_time_field(), ref)
