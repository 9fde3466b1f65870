"""Unequal spacings so far apart, or so large, that the roots' range tests are
needed although h s along x is ordinary: the default solve is the oracle's,
bit for bit."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("d,s0", [
    # the y-z plane's determinants near 2^-980
    ((1.0, 2.0 ** -250, 1.25 * 2.0 ** -251), 2.0 ** -240),
    # the 3D determinant, of the size of (s / h)^2, near 2^-996
    ((2.0 ** 200, 1.5 * 2.0 ** 200, 1.25 * 2.0 ** 200), 2.0 ** -299),
    # in range
    ((10.0, 12.5, 8.0), 1.0 / 3000.0)])
@pytest.mark.parametrize("radius", [-1, 2])
def test_default_solve_is_the_oracles(ekx, oracle, d, s0, radius):
    dims = (13, 10, 12)
    rng = np.random.default_rng(3)
    slow = s0 * rng.uniform(0.5, 1.5, 12 * 9 * 11)
    # on a plane of nodes in x, where the times of y and z count alone
    src = (5 * d[0], 0.4 * 9 * d[1], 0.4 * 11 * d[2])
    print("case", d, s0, radius, flush=True)
    s = ekx.Solver3D()
    s.initialize(ekx.SolverOptions(number_of_sweeps=2,
                                   factored_radius=radius),
                 ekx.Geometry3D(*dims, *d))
    s.set_slowness(slow)
    s.set_source(src)
    s.solve()
    ref = oracle.solve3d(oracle.geometry3d(*dims, *d), slow, src, 2, radius)
    got = s.get_travel_time_field()
    print("differ", int((got != ref).sum()), "of", ref.size, flush=True)
    assert np.array_equal(got, ref)
