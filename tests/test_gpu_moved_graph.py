"""Solves whose captured launches do not depend on the source keep their graph
when the source moves (no factored box).  Each field is the oracle's, and a
solve after a move takes no longer than one after none: capturing the 13440
launches again adds 17% to its time; the bar is 8%, of the shortest of nine."""
import time

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def test_graph_kept_when_it_does_not_depend_on_the_source(ekx, oracle):
    dims, h, sweeps, n = (17, 17, 64), 10.0, 20, 16
    rng = np.random.default_rng(6)
    slow = 1.0 / rng.uniform(1800.0, 5200.0, 16 * 16 * 63)
    sources = [(25.0, 31.0, 44.0), (131.0, 102.0, 625.0)]
    g = ekx.Geometry3D(*dims, h)
    b = ekx.Batch3D()
    b.initialize(ekx.SolverOptions(
        number_of_sweeps=sweeps, factored_radius=-1, chunk_planes=64,
        chains=n, launch_order=ekx.LaunchOrder.DIAGONALS),
        [(g, slow, sources[0])] * n)
    refs = [oracle.solve3d(oracle.geometry3d(*dims, h), slow, x, sweeps, -1)
            for x in sources]
    times = {True: [], False: []}
    for k in range(22):
        at = (k + 1) // 2 % 2       # sources 0, 1, 1, 0, 0, 1, ...
        for i in range(n):
            b.set_source(i, sources[at])
        t = time.perf_counter()
        b.solve()
        if k >= 4:
            times[k % 2 == 1].append(time.perf_counter() - t)
        for i in (0, n - 1):
            assert np.array_equal(b.get_travel_time_field(i), refs[at]), k
    moved, kept = min(times[True]), min(times[False])
    print("moved %.2f ms, not moved %.2f ms" % (1e3 * moved, 1e3 * kept),
          flush=True)
    assert moved <= 1.08 * kept
