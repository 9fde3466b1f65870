"""Solves by launches per diagonal, named where the default is one launch: the
captured graph against eager launches, the tuned shape, the size-class default
depths, and FP64 chunks of 64 to 79 planes with the factored box inside and a
source that moves."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _slow(dims, seed):
    rng = np.random.default_rng(seed)
    return rng, 1.0 / rng.uniform(1800.0, 5200.0, (dims[0] - 1)
                                  * (dims[1] - 1) * (dims[2] - 1))


def _solver(ekx, dims, h, slow, precision="FP64", **options):
    s = ekx.Solver3D()
    s.initialize(ekx.SolverOptions(
        factored_radius=3, launch_order=ekx.LaunchOrder.DIAGONALS,
        precision=getattr(ekx.Precision, precision), **options),
        ekx.Geometry3D(*dims, h))
    s.set_slowness(slow)
    return s


@pytest.mark.parametrize("precision", ["FP64", "FP32_POLISH", "FIXED32"])
@pytest.mark.parametrize("chunk", [0, 66])
def test_graph_and_eager_agree(ekx, oracle, precision, chunk):
    dims, h = (41, 33, 66), 10.0
    _, slow = _slow(dims, 1)
    ref = {}
    for use_graph in (True, False):
        s = _solver(ekx, dims, h, slow, precision, number_of_sweeps=2,
                    chunk_planes=chunk, use_graph=use_graph)
        for k, src in enumerate([(55.0, 60.0, 77.0), (390.0, 20.0, 600.0),
                                 (55.0, 60.0, 77.0)]):
            print("case", precision, chunk, use_graph, k, flush=True)
            s.set_source(src)
            s.solve()
            assert s.get_stats().kernel_launches > 24
            got = s.get_travel_time_field()
            assert np.array_equal(got, ref.setdefault(src, got))
            if precision == "FP64":
                assert np.array_equal(got, oracle.solve3d(
                    oracle.geometry3d(*dims, h), slow, src, 2, 3))


@pytest.mark.parametrize("precision", ["FP64", "FP32_POLISH", "FIXED32"])
def test_tuned_shape_runs(ekx, precision):
    dims, h = (41, 33, 66), 10.0
    _, slow = _slow(dims, 2)
    src = (123.0, 45.0, 321.0)
    s = _solver(ekx, dims, h, slow, precision, number_of_sweeps=2)
    s.set_source(src)
    s.solve()
    ref = s.get_travel_time_field()
    chunk, chains = s.autotune()
    s.solve()
    st = s.get_stats()
    print("tuned", chunk, chains, st.kernel_launches, flush=True)
    assert (st.chunk_planes, st.chains) == (chunk, chains)
    # one iteration or more of 8 sweeps after 8, each a launch per diagonal
    diagonals = 6 + 5 + -(-66 // chunk) - 2
    assert st.kernel_launches >= 24 * diagonals
    assert np.array_equal(s.get_travel_time_field(), ref)


@pytest.mark.parametrize("precision", ["FP64", "FP32_POLISH", "FIXED32"])
@pytest.mark.parametrize("dims", [(9, 8, 3), (25, 31, 8), (17, 40, 41)])
def test_default_depths(ekx, oracle, precision, dims):
    _, slow = _slow(dims, 3)
    src = tuple(0.3 * (n - 1) * 10.0 for n in dims)
    out = []
    for chunk in (0, 5):
        s = _solver(ekx, dims, 10.0, slow, precision, number_of_sweeps=2,
                    chunk_planes=chunk)
        s.set_source(src)
        s.solve()
        assert s.get_stats().kernel_launches > 2
        out.append(s.get_travel_time_field())
    assert np.array_equal(*out)
    if precision == "FP64":
        assert np.array_equal(out[0], oracle.solve3d(
            oracle.geometry3d(*dims, 10.0), slow, src, 2, 3))


def test_box_inside_deep_chunks(ekx, oracle):
    """3000 problems of 16 x 16 x 70: whole columns of 70 planes by default,
    their box in the bulk launches, replayed after the sources have moved."""
    dims, h, n = (16, 16, 70), 10.0, 3000
    rng, slow = _slow(dims, 4)
    g = ekx.Geometry3D(*dims, h)

    def draw():
        return [tuple(float(rng.uniform(0, (m - 1) * h)) for m in dims)
                for _ in range(n)]
    sources = draw()
    b = ekx.Batch3D()
    b.initialize(ekx.SolverOptions(
        number_of_sweeps=1, factored_radius=3,
        launch_order=ekx.LaunchOrder.DIAGONALS),
        [(g, slow, x) for x in sources])
    for move in range(2):
        if move:
            sources = draw()
            for i, x in enumerate(sources):
                b.set_source(i, x)
        b.solve()
        st = b.get_stats()
        print("case", move, st.as_dict(), flush=True)
        assert st.chunk_planes == 70
        for i in (0, 1, 1500, 2998, 2999):
            ref = oracle.solve3d(oracle.geometry3d(*dims, h), slow,
                                 sources[i], 1, 3)
            assert np.array_equal(b.get_travel_time_field(i), ref), (move, i)
