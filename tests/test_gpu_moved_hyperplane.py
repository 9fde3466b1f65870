"""A source that moves between solves of the hyperplane kernel, whose captured
launches hold each level's extent, which follows the source's octants: every
solve is the oracle's."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("batch", [False, True])
def test_levels_follow_the_source(ekx, oracle, batch):
    dims, h = (21, 17, 26), 10.0
    rng = np.random.default_rng(4)
    slow = 1.0 / rng.uniform(1800.0, 5200.0, 20 * 16 * 25)
    options = ekx.SolverOptions(number_of_sweeps=1, factored_radius=2,
                                kernel=ekx.Kernel.HYPERPLANE)
    sources = [(195.0, 5.0, 245.0), (5.0, 155.0, 5.0), (104.0, 83.0, 120.0),
               (195.0, 5.0, 245.0)]
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
        ref = oracle.solve3d(oracle.geometry3d(*dims, h), slow, src, 1, 2)
        assert np.array_equal(field, ref), src
