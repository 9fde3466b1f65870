"""Models on both sides of the square roots' range rules: slownesses whose
h s are ordinary, and so small that h s h s leaves the range in which the
roots need no scaling (h s about 2^-340 and 2^-400: the 3D rule's and the 2D
rule's other side), on short chunks, whole columns and in 2D.  The 3D field
equals the oracle's bit for bit on either route; the 2D one to the 2D
solver's bar of 1e-12."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("exponent", [0, -330, -390])
@pytest.mark.parametrize("chunk", [0, 7, 70])
def test_3d(ekx, oracle, exponent, chunk):
    nx, ny, nz, h = 19, 11, 72, 10.0
    rng = np.random.default_rng(91)
    slow = (1.0 / rng.uniform(2000.0, 4000.0, (nx - 1) * (ny - 1) * (nz - 1))
            * 2.0**exponent)
    src = (81.0, 44.0, 333.0)
    print("case", exponent, chunk, flush=True)
    s = ekx.Solver3D()
    s.initialize(ekx.SolverOptions(number_of_sweeps=2, factored_radius=2,
                                   chunk_planes=chunk),
                 ekx.Geometry3D(nx, ny, nz, h))
    s.set_slowness(slow)
    s.set_source(src)
    s.solve()
    ref = oracle.solve3d(oracle.geometry3d(nx, ny, nz, h), slow, src, 2, 2)
    assert np.array_equal(s.get_travel_time_field(), ref)


@pytest.mark.parametrize("exponent", [0, -330, -390])
@pytest.mark.parametrize("dz", [10.0, 12.5])
def test_2d(ekx, oracle, exponent, dz):
    nx, nz, dx = 40, 70, 10.0
    rng = np.random.default_rng(92)
    slow = (1.0 / rng.uniform(2000.0, 4000.0, (nx - 1) * (nz - 1))
            * 2.0**exponent)
    src = (181.0, 333.0)
    print("case", exponent, dz, flush=True)
    s = ekx.Solver2D()
    s.initialize(ekx.SolverOptions(number_of_sweeps=2, factored_radius=2),
                 ekx.Geometry2D(nx, nz, dx, dz))
    s.set_slowness(slow)
    s.set_source(src)
    s.solve()
    got = s.get_travel_time_field()
    ref = oracle.solve2d(oracle.geometry2d(nx, nz, dx, dz), slow, src, 2, 2)
    rel = np.abs(got - ref) / np.maximum(ref, slow.min() * dx)
    print("max rel", rel.max())
    assert rel.max() <= 1e-12
