"""The 2D band kernel at the edges of its bands, groups and range: rows
around multiples of 64 (one lane, a full band, a band of one row), columns
around multiples of the 8-step groups, the tallest grid it takes and one
beyond it (the level kernel), both operators, sources in corners and
centres; against the oracle.

The kernel keeps the oracle's operation order, so every operation outside
the factored box rounds alike; inside it hypot may differ by an ulp of the
analytic time, which the box's own square roots of near-zero discriminants
can magnify: the repository's 1e-12 relative bar of the 2D solver."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SHAPES = [(3, 3), (5, 64), (8, 65), (9, 63), (64, 66), (65, 128), (71, 129),
          (130, 7), (40, 200), (17, 1024), (12, 1025)]


@pytest.mark.parametrize("nx,nz", SHAPES)
@pytest.mark.parametrize("dz", [10.0, 12.5])
def test_band_edges(ekx, oracle, nx, nz, dz):
    dx = 10.0
    rng = np.random.default_rng(nx * 7919 + nz)
    slow = 1.0 / rng.uniform(1500.0, 5500.0, (nx - 1) * (nz - 1))
    ext = ((nx - 1) * dx, (nz - 1) * dz)
    sources = [(0.0, 0.0), ext, (0.37 * ext[0], 0.61 * ext[1])]
    for k, (src, radius, sweeps) in enumerate(
            zip(sources, (3, 2, -1), (1, 0, 2))):
        print("case", nx, nz, dz, k, flush=True)
        s = ekx.Solver2D()
        s.initialize(ekx.SolverOptions(number_of_sweeps=sweeps,
                                       factored_radius=radius),
                     ekx.Geometry2D(nx, nz, dx, dz))
        s.set_slowness(slow)
        s.set_source(src)
        for _ in range(2):          # a second solve on the used buffers
            s.solve()
            got = s.get_travel_time_field()
            ref = oracle.solve2d(oracle.geometry2d(nx, nz, dx, dz), slow,
                                 src, sweeps, radius)
            rel = np.abs(got - ref) / np.maximum(ref, slow.min() * dx)
            print("max rel", rel.max(), flush=True)
            assert rel.max() <= 1e-12
