"""The band kernel's instances by rows: 512 (8 waves, read 8 steps ahead), 513 to
768 (12 waves, 4 ahead: a group of 8 steps in two parts) and 769 on (16, 2
ahead), at their edges and inside; against the oracle with the 2D solver's bar
of 1e-12 (hypot's ulp in the factored box)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx,nz", [(9, 512), (11, 513), (70, 523), (8, 576),
                                   (13, 577), (30, 640), (10, 768), (9, 769),
                                   (24, 900)])
@pytest.mark.parametrize("dz", [10.0, 12.5])
def test_rows(ekx, oracle, nx, nz, dz):
    rng = np.random.default_rng(nx * 7919 + nz)
    slow = 1.0 / rng.uniform(1500.0, 5500.0, (nx - 1) * (nz - 1))
    ext = ((nx - 1) * 10.0, (nz - 1) * dz)
    for k, (src, radius, sweeps) in enumerate(zip(
            [(0.0, 0.0), ext, (0.37 * ext[0], 0.61 * ext[1])],
            (3, 2, -1), (1, 0, 2))):
        print("case", nx, nz, dz, k, flush=True)
        s = ekx.Solver2D()
        s.initialize(ekx.SolverOptions(number_of_sweeps=sweeps,
                                       factored_radius=radius),
                     ekx.Geometry2D(nx, nz, 10.0, dz))
        s.set_slowness(slow)
        s.set_source(src)
        ref = oracle.solve2d(oracle.geometry2d(nx, nz, 10.0, dz), slow, src,
                             sweeps, radius)
        for _ in range(2):
            s.solve()
            rel = np.abs(s.get_travel_time_field() - ref) / np.maximum(
                ref, slow.min() * 10.0)
            assert rel.max() <= 1e-12
