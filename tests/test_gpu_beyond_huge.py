"""Models so slow that times at the source cell's corners exceed HUGE (1e10), the
start value of every other node: a candidate that is not valid counts as
HUGE, neither more nor less.  2D against the oracle, 3D the default solve
against the launches per diagonal."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx,nz", [(9, 12), (8, 65), (11, 130), (6, 1030)])
@pytest.mark.parametrize("dz", [10.0, 12.5])
@pytest.mark.parametrize("s0", [1e8, 3e9, 1e11])
def test_2d(ekx, oracle, nx, nz, dz, s0):
    rng = np.random.default_rng(nx + nz)
    slow = s0 * rng.uniform(0.5, 2.0, (nx - 1) * (nz - 1))
    src = (0.4 * (nx - 1) * 10.0, 0.7 * (nz - 1) * dz)
    print("case", nx, nz, dz, s0, flush=True)
    for radius, sweeps in ((3, 1), (-1, 2)):
        s = ekx.Solver2D()
        s.initialize(ekx.SolverOptions(number_of_sweeps=sweeps,
                                       factored_radius=radius),
                     ekx.Geometry2D(nx, nz, 10.0, dz))
        s.set_slowness(slow)
        s.set_source(src)
        s.solve()
        got = s.get_travel_time_field()
        ref = oracle.solve2d(oracle.geometry2d(nx, nz, 10.0, dz), slow, src,
                             sweeps, radius)
        rel = np.abs(got - ref) / ref
        print("differ", int((rel > 1e-12).sum()), rel.max(), flush=True)
        assert rel.max() <= 1e-12


@pytest.mark.parametrize("d", [(10.0, 10.0, 10.0), (10.0, 12.5, 8.0)])
@pytest.mark.parametrize("s0", [1e8, 3e9, 1e11])
@pytest.mark.parametrize("precision", ["FP64", "FP32_POLISH"])
def test_3d(ekx, d, s0, precision):
    dims = (19, 10, 12)
    rng = np.random.default_rng(5)
    slow = s0 * rng.uniform(0.5, 2.0, 18 * 9 * 11)
    src = tuple(0.43 * (n - 1) * h for n, h in zip(dims, d))
    for radius in (-1, 2):
        print("case", d, s0, precision, radius, flush=True)
        out = []
        for chunk in (0, 8):
            s = ekx.Solver3D()
            s.initialize(ekx.SolverOptions(
                number_of_sweeps=2, factored_radius=radius,
                chunk_planes=chunk,
                precision=getattr(ekx.Precision, precision)),
                ekx.Geometry3D(*dims, *d))
            s.set_slowness(slow)
            s.set_source(src)
            s.solve()
            out.append(s.get_travel_time_field())
        print("differ", int((out[0] != out[1]).sum()), flush=True)
        assert np.array_equal(*out)
