"""A source that moves between solves: the launches of the factored box on
its own diagonals (deep chunks) follow it, also where a captured graph is
replayed."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("batch", [False, True])
def test_factored_launches_follow_the_source(ekx, oracle, batch):
    dims, h = (40, 24, 70), 10.0
    rng = np.random.default_rng(2)
    slow = 1.0 / rng.uniform(1800.0, 5200.0, 39 * 23 * 69)
    options = ekx.SolverOptions(number_of_sweeps=1, factored_radius=3,
                                chunk_planes=70)
    sources = [(25.0, 31.0, 44.0), (371.0, 202.0, 655.0), (25.0, 31.0, 44.0)]
    g = ekx.Geometry3D(*dims, h)
    if batch:
        s = ekx.Batch3D()
        s.initialize(options, [(g, slow, sources[0])])
    else:
        s = ekx.Solver3D()
        s.initialize(options, g)
        s.set_slowness(slow)
    for src in sources:
        print("case", batch, src, flush=True)
        s.set_source(*((0, src) if batch else (src,)))
        s.solve()
        field = s.get_travel_time_field(*((0,) if batch else ()))
        ref = oracle.solve3d(oracle.geometry3d(*dims, h), slow, src, 1, 3)
        assert np.array_equal(field, ref), src
