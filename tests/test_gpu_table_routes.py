"""Which kernel a launch of the tabulated problem takes, by its paths and by whether the stencils'
tiles fit in LDS (counters.wg_size: 256 several lanes to a path, 512 tiled, the run's own otherwise),
and that each gives the same bits; FP64 knots are the oracle's."""
import numpy as np
import pytest

from oracle import oracle as O

pytestmark = pytest.mark.gpu
SW, NE = (-1.0, -1.0), (1.0, 1.0)
BOX = SW + NE


@pytest.fixture(scope="module")
def eng():
    from pdds_amd.engine import Engine
    e = Engine(0)
    yield e
    e.close()


@pytest.fixture(scope="module")
def mesh():
    from pdds_amd.engine import Mesh
    from pdds_amd.workloads import relative_fac
    return Mesh(SW, NE, 4, 8, relative_fac(SW, NE, 4, 8, 0.8))


def _problem(eng, n, nv):
    """The tables on n x n texels, those of mu and F on nv x nv."""
    from pdds_amd import workloads as W
    from pdds_amd.engine import bvp
    grid = {k: np.meshgrid(np.linspace(-1, 1, k), np.linspace(-1, 1, k)) for k in (n, nv)}
    f, u, v = W.varcoef_table_fields(*grid[n]), W.varcoef_u(*grid[n]), W.varcoef_vrcv_fields(*grid[nv], 0.5)
    return (bvp("table", lut=eng.lut(f, BOX), ulut=eng.lut(u, BOX), vlut=eng.lut(v, BOX)),
            (O.lut_dict(f, BOX), O.lut_dict(u, BOX), O.lut_dict(v, BOX)))


def _run(eng, mesh, prob, counts, **run):
    from pdds_amd.engine import default_run
    return eng.assemble(mesh, prob, default_run(wg_size=128, sub_batch=32, item_paths=640, **run), 0, paths_per_knot=counts)


def _counts(mesh, per_lane, cu):
    """Counts of a launch of a little more than per_lane paths per lane of the tiled grid."""
    n = np.where(mesh.on_boundary, 0, per_lane * cu * 512 // int(np.sum(~mesh.on_boundary)) + 20).astype(np.int64)
    n[70] = 1437
    return n


def _same(a, b):
    for k in ("G", "Gvar", "B", "BB"):
        assert np.array_equal(a[k], b[k]), k
    for k in ("path_steps", "paths", "exits"):
        assert a["counters"][k] == b["counters"][k], k


# 64: every tile with three planes; 64 with another grid of mu and F: two planes
@pytest.mark.parametrize("n,nv", [(64, 64), (64, 50)])
@pytest.mark.parametrize("precision,step", [("fp64", 0), ("fp64", 1), ("fp64", 2), ("fp64", 3), ("fp32", 0), ("fp32", 1),
                                            ("fp32", 2), ("fp32", 3)])
def test_tiled_equals_persistent_and_oracle(eng, mesh, n, nv, precision, step):
    prob, (fl, ul, vl) = _problem(eng, n, nv)
    cu = eng.info()["n_cu"]
    run = dict(h=8e-3, seed=9, step=step, precision=precision)
    print("table", n, nv, precision, step, flush=True)
    got = _run(eng, mesh, prob, _counts(mesh, 5, cu), **run)
    ref = _run(eng, mesh, prob, _counts(mesh, 5, cu), lut_lds=0, **run)
    # (the FP32 VR and VR + CV steps have no tiled form)
    assert got["counters"]["wg_size"] == (128 if precision == "fp32" and step >= 2 else 512)
    assert ref["counters"]["wg_size"] == 128
    _same(got, ref)
    few = _run(eng, mesh, prob, _counts(mesh, 3, cu), **run)
    assert few["counters"]["wg_size"] == 128
    knot, c = 70, 1437
    r = slice(mesh.row_ptr[knot], mesh.row_ptr[knot + 1])
    assert np.array_equal(few["G"][r], got["G"][r]) and few["B"][knot] == got["B"][knot]
    if precision == "fp64":
        from pdds_amd.workloads import relative_fac
        fac = relative_fac(SW, NE, 4, 8, 0.8)
        st = mesh.stencil(knot)
        pb = O.problem(O.PDE_TABLE, lut=fl, ulut=ul, vlut=vl, step=step)
        paths = O.simulate(pb, O.run_params(8e-3, 9, threads=8), mesh.x0[knot], mesh.y0[knot], st["rect"], knot, 0, c)
        o = O.reduce_batched(pb, paths, st, mesh.glob, [fac[min(max(int(v), 0), 3)] for v in st["kind"]], st["ipsi"],
                             32, 640, quirk=1)
        assert got["B"][knot] == o["B"] and got["BB"][knot] == o["BB"] and np.array_equal(got["G"][r], o["G"])


# no tile fits; the crossings' do not
@pytest.mark.parametrize("n,per_lane,wg", [(600, 5, 128), (600, 40, 128), (160, 5, 128), (160, 40, 512)])
@pytest.mark.parametrize("precision", ["fp64", "fp32"])
def test_launches_whose_tiles_do_not_all_fit(eng, n, per_lane, wg, precision):
    from pdds_amd.engine import Mesh
    from pdds_amd.workloads import relative_fac, table_problem
    m = Mesh(SW, NE, 4, 16, relative_fac(SW, NE, 4, 16, 0.8))
    counts = _counts(m, per_lane, eng.info()["n_cu"])
    print("table", n, per_lane, precision, flush=True)
    run = dict(h=1e-2, seed=4, precision=precision)
    got = _run(eng, m, table_problem(eng, n, BOX), counts, **run)
    assert got["counters"]["wg_size"] == wg
    _same(got, _run(eng, m, table_problem(eng, n, BOX), counts, lut_lds=0, **run))


@pytest.mark.parametrize("precision,most", [("fp64", 512), ("fp32", 256)])
def test_few_paths_run_several_lanes_to_a_path(eng, precision, most):
    """On both sides of the limit, per CU; the points they share are equal."""
    from pdds_amd.engine import default_run
    from pdds_amd.workloads import table_problem
    cu = eng.info()["n_cu"]
    prob = table_problem(eng, 64, BOX)
    x, y, out = np.array([0.1, -0.6, 0.4]), np.array([-0.3, 0.2, 0.9]), []
    for last, wg in ((cu * most - 3041, 256), (cu * most - 3040, 128)):
        r = eng.point_eval(prob, default_run(h=1e-2, seed=9, precision=precision, wg_size=128), np.array(BOX), x, y,
                           np.array([3000, 41, last]))
        assert r["counters"]["wg_size"] == wg
        out.append((r["u"][:2], r["u_var"][:2]))
    assert np.array_equal(out[0][0], out[1][0]) and np.array_equal(out[0][1], out[1][1])
