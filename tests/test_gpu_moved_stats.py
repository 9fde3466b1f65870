"""Work counts after a source has moved: those of a solver that starts there,
also where a captured graph is replayed."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", ["FP64", "FIXED32", "FP32_POLISH"])
@pytest.mark.parametrize("order,chunk", [
    ("DIAGONALS", 0), ("DIAGONALS", 8), ("DIAGONALS", 70), ("AUTO", 0)])
def test_counts_follow_the_source(ekx, precision, order, chunk):
    dims, h = (40, 24, 70), 10.0
    slow = np.full(39 * 23 * 69, 1.0 / 3000.0)
    sources = [(25.0, 31.0, 44.0), (371.0, 202.0, 655.0), (201.0, 99.0, 8.0)]

    def make():
        s = ekx.Solver3D()
        s.initialize(ekx.SolverOptions(
            number_of_sweeps=2, factored_radius=3, chunk_planes=chunk,
            precision=getattr(ekx.Precision, precision),
            launch_order=getattr(ekx.LaunchOrder, order)),
            ekx.Geometry3D(*dims, h))
        s.set_slowness(slow)
        return s
    moving = make()
    for k, src in enumerate([*sources, sources[0]]):
        if k == 3:
            moving.autotune()       # (another depth may count other boxes)
        counts = []
        for s in (moving, make()):
            s.set_source(src)
            s.solve()
            st = s.get_stats()
            counts.append([st.updates, st.updates_fp64, st.iterations_run])
            if k < 3:
                counts[-1] += [st.updates_factored, st.kernel_launches]
        print("case", precision, order, chunk, src, counts, flush=True)
        assert counts[0] == counts[1]
