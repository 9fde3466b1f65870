"""2D solvers, 2D batches, generated models, a second 3D solver and the device's
synchronisation on one thread while another captures the launches of a 3D
solver: neither disturbs the other."""
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def test_2d_beside_a_capture(ekx, oracle):
    dims, h, n = (17, 17, 70), 10.0, 16
    rng = np.random.default_rng(6)
    slow3 = 1.0 / rng.uniform(1800.0, 5200.0, 16 * 16 * 69)
    g3 = ekx.Geometry3D(*dims, h)
    sources = [(25.0, 31.0, 44.0), (131.0, 102.0, 655.0)]
    refs = [oracle.solve3d(oracle.geometry3d(*dims, h), slow3, x, 4, 2)
            for x in sources]
    stop, trouble, rounds = threading.Event(), [], [0, 0]

    def capture():
        try:
            b = ekx.Batch3D()
            b.initialize(ekx.SolverOptions(
                number_of_sweeps=4, factored_radius=2, chunk_planes=70,
                chains=n, launch_order=ekx.LaunchOrder.DIAGONALS),
                [(g3, slow3, sources[0])] * n)
            while not stop.is_set():
                src = rounds[0] % 2
                for i in range(n):
                    b.set_source(i, sources[src])
                b.solve()
                assert np.array_equal(b.get_travel_time_field(n - 1),
                                      refs[src])
                rounds[0] += 1
        except Exception as e:      # (raised again below)
            trouble.append(e)

    slow2 = 1.0 / rng.uniform(1500.0, 5500.0, 40 * 50)
    g2 = ekx.Geometry2D(41, 51, 10.0)
    src2 = (123.0, 321.0)
    ref2 = oracle.solve2d(oracle.geometry2d(41, 51, 10.0, 10.0), slow2, src2,
                          1, 3)
    o = ekx.SolverOptions(number_of_sweeps=1, factored_radius=3)

    def same(field):
        rel = np.abs(field - ref2) / np.maximum(ref2, slow2.min() * 10.0)
        assert rel.max() <= 1e-12

    small = (9, 11, 10)
    slow_small = 1.0 / rng.uniform(1800.0, 5200.0, 8 * 10 * 9)
    s3 = ekx.Solver3D()
    s3.initialize(ekx.SolverOptions(number_of_sweeps=1, factored_radius=2),
                  ekx.Geometry3D(*small, h))
    s3.set_slowness(slow_small)
    s3.set_stations([(20.0, 30.0, 40.0)])
    ref3 = oracle.solve3d(oracle.geometry3d(*small, h), slow_small,
                          (31.0, 22.0, 13.0), 1, 2)
    model = ekx.LayeredGaussianModel([2500.0, 3500.0, 5000.0], 0.1, 40.0, 2)
    gm = ekx.Geometry3D(20, 9, 13, 5.0, 12.0, 7.0)
    velocity = model.generate(gm)
    thread = threading.Thread(target=capture)
    thread.start()
    try:
        s = ekx.Solver2D()
        s.initialize(o, g2)
        s.set_slowness(slow2)
        while rounds[0] < 12 and thread.is_alive():
            s.set_source(src2)
            s.set_stations([(10.0, 20.0), (300.0, 400.0)])
            s.solve()
            same(s.get_travel_time_field())
            assert len(s.get_travel_times_at_stations()) == 2
            s.compute_travel_time_gradient_field()
            s.get_travel_time_gradient_field()
            assert np.array_equal(model.generate(gm), velocity)
            ekx.synchronize()
            s3.set_source((31.0, 22.0, 13.0))
            s3.solve()
            assert np.array_equal(s3.get_travel_time_field(), ref3)
            assert len(s3.get_travel_times_at_stations()) == 1
            s3.compute_travel_time_gradient_field()
            s3.get_travel_time_gradient_field()
            b = ekx.Batch2D()
            b.initialize(o, [(g2, slow2, src2)] * 3)
            b.solve()
            same(b.get_travel_time_field(2))
            rounds[1] += 1
    finally:
        stop.set()
        thread.join()
    print("rounds", rounds, flush=True)
    assert not trouble, trouble
    assert rounds[0] >= 12 and rounds[1] > 0
