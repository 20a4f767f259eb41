"""Which kernel a launch of the coefficient-LUT problem takes, by its paths and by whether the
stencils' tiles fit in LDS (counters.wg_size: 256 several lanes to a path, 512 or 768 tiled, the
run's own otherwise), on both sides of each limit.  The knots that two launches share are equal."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
SW, NE = (-1.0, -1.0), (1.0, 1.0)
BOX = SW + NE


@pytest.fixture(scope="module")
def eng():
    from pdds_amd.engine import Engine
    e = Engine(0)
    yield e
    e.close()


def _counts(mesh, total):
    """About `total` paths (never fewer), 1237 of them at the second interior knot."""
    inner = np.flatnonzero(~mesh.on_boundary)
    n = np.zeros(mesh.n_knots, dtype=np.int64)
    n[inner] = -(-(total - 1237) // (len(inner) - 1))
    n[inner[1]] = 1237
    return n, int(inner[1])


# samples per side: 64 every tile fits, 256 the crossing's does not, 512 none; paths per CU at the limit
@pytest.mark.parametrize("precision,n,per_cu,wg", [("fp64", 64, 24 * 512, 512), ("fp64", 512, 24 * 512, 512),
                                                   ("fp32", 64, 4 * 768, 768), ("fp32", 256, 16 * 768, 768),
                                                   ("fp32", 512, 16 * 768, 128)])
def test_tiles_by_paths_and_fit(eng, precision, n, per_cu, wg):
    from pdds_amd.engine import Mesh, bvp, default_run
    from pdds_amd.workloads import relative_fac, varcoef_lut
    m = Mesh(SW, NE, 4, 16, relative_fac(SW, NE, 4, 16, 0.8))
    prob, total = bvp("varcoef_lut", lut=varcoef_lut(eng, n, BOX)), per_cu * eng.info()["n_cu"]
    run = dict(h=1e-2, seed=9, precision=precision, wg_size=128, sub_batch=32, item_paths=640)
    out = []
    for paths, want in ((total - 1000, 128), (total, wg)):
        c, knot = _counts(m, paths)
        if want == 128 and paths < total:
            c[np.flatnonzero(~m.on_boundary)[2]] -= max(0, int(c.sum()) - paths)
        print(precision, n, int(c.sum()), flush=True)
        got = eng.assemble(m, prob, default_run(**run), 0, paths_per_knot=c)
        assert got["counters"]["wg_size"] == want
        r = slice(m.row_ptr[knot], m.row_ptr[knot + 1])
        out.append((got["G"][r], got["B"][knot], got["BB"][knot]))
    assert np.array_equal(out[0][0], out[1][0]) and out[0][1:] == out[1][1:]


@pytest.mark.parametrize("precision,most", [("fp64", 384), ("fp32", 256)])
def test_few_paths_run_several_lanes_to_a_path(eng, precision, most):
    from pdds_amd.engine import bvp, default_run
    from pdds_amd.workloads import varcoef_lut
    cu = eng.info()["n_cu"]
    prob = bvp("varcoef_lut", lut=varcoef_lut(eng, 64, BOX))
    x, y, out = np.array([0.1, -0.6, 0.4]), np.array([-0.3, 0.2, 0.9]), []
    for last, wg in ((cu * most - 3041, 256), (cu * most - 3040, 128)):
        r = eng.point_eval(prob, default_run(h=1e-2, seed=9, precision=precision, wg_size=128), np.array(BOX), x, y,
                           np.array([3000, 41, last]))
        assert r["counters"]["wg_size"] == wg
        out.append((r["u"][:2], r["u_var"][:2]))
    assert np.array_equal(out[0][0], out[1][0]) and np.array_equal(out[0][1], out[1][1])
