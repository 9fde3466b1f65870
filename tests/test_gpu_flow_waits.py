"""Waits of the one-launch solves: their bound follows the number of sweeps
where problems wait for others to finish."""
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
