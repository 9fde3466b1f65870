"""The default depth of the column chunks by element type: whole columns of 193
planes from 2.5 (FP64), 3.5 (scaled integers) and 4 (FP32) times the
resident waves a diagonal on, half columns below.  Fields do not depend on it."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision,n,chunk", [
    ("FP64", 2700, 97), ("FP64", 3600, 193), ("FIXED32", 3600, 97),
    ("FIXED32", 4200, 193), ("FP32", 3600, 97), ("FP32", 4200, 97),
    ("FP32", 5800, 193)])
def test_default_depth(ekx, precision, n, chunk):
    """17 x 17 x 193: 9 columns on 5 diagonals a problem, 2048 resident
    waves."""
    dims, h = (17, 17, 193), 10.0
    slow = 1.0 / np.random.default_rng(1).uniform(2000.0, 5000.0,
                                                  16 * 16 * 192)
    g = ekx.Geometry3D(*dims, h)
    sources = [(31.0 + 0.01 * i, 44.0, 905.0) for i in range(n)]
    print("case", precision, n, flush=True)
    b = ekx.Batch3D()
    b.initialize(ekx.SolverOptions(
        number_of_sweeps=0, factored_radius=2,
        precision=getattr(ekx.Precision, precision),
        launch_order=ekx.LaunchOrder.DIAGONALS),
        [(g, slow, x) for x in sources])
    b.solve()
    assert b.get_stats().chunk_planes == chunk
    one = ekx.Batch3D()
    one.initialize(ekx.SolverOptions(
        number_of_sweeps=0, factored_radius=2, chunk_planes=8,
        precision=getattr(ekx.Precision, precision)),
        [(g, slow, sources[n - 1])])
    one.solve()
    assert np.array_equal(b.get_travel_time_field(n - 1),
                          one.get_travel_time_field(0))
