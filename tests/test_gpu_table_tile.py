"""The tabulated problem in the LDS-tiled path kernel: launches of at least one path per lane of its
grid (131072 on 256 CUs).  The tile holds two planes, three with the VR + CV step where the second
table has the same grid and there is room, none for the stencils it does not fit; the results are
those of the persistent kernel (lut_lds 0), and one knot's the oracle's, bit for bit."""
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


def _problem(eng, n, nv):
    """The tables on n x n texels, those of mu and F on nv x nv."""
    from pdds_amd import workloads as W
    from pdds_amd.engine import bvp
    grid = {k: np.meshgrid(np.linspace(-1, 1, k), np.linspace(-1, 1, k)) for k in (n, nv)}
    f, u, v = W.varcoef_table_fields(*grid[n]), W.varcoef_u(*grid[n]), W.varcoef_vrcv_fields(*grid[nv], 0.5)
    prob = bvp("table", lut=eng.lut(f, BOX), ulut=eng.lut(u, BOX), vlut=eng.lut(v, BOX))
    return prob, (O.lut_dict(f, BOX), O.lut_dict(u, BOX), O.lut_dict(v, BOX))


# 64: every tile fits with three planes; 160: some with three, some with two; 300: some with none
@pytest.mark.parametrize("n,nv", [(64, 64), (64, 50), (160, 160), (300, 300)])
@pytest.mark.parametrize("precision,step", [("fp64", 0), ("fp64", 1), ("fp64", 2), ("fp64", 3), ("fp32", 0),
                                            ("fp32", 1), ("fp32", 2), ("fp32", 3)])
def test_tiled_equals_persistent_and_oracle(eng, n, nv, precision, step):
    from pdds_amd.engine import Mesh, default_run
    from pdds_amd.workloads import relative_fac
    prob, (fl, ul, vl) = _problem(eng, n, nv)
    fac = relative_fac(SW, NE, 4, 8, 0.8)
    m = Mesh(SW, NE, 4, 8, fac)
    counts = np.where(m.on_boundary, 1, 1500).astype(np.int64)
    counts[70] = 1437
    # FP64 launches with the control-variate step of up to 2048 paths per CU go to another kernel
    if step == 0:
        counts[~m.on_boundary] *= 4
    run = dict(h=2e-3, seed=9, step=step, precision=precision, sub_batch=32, item_paths=640)
    got = eng.assemble(m, prob, default_run(lut_lds=1, **run), 1500, paths_per_knot=counts)
    ref = eng.assemble(m, prob, default_run(lut_lds=0, **run), 1500, paths_per_knot=counts)
    for k in ("G", "Gvar", "B", "BB"):
        assert np.array_equal(got[k], ref[k]), k
    assert got["counters"]["path_steps"] == ref["counters"]["path_steps"]
    if precision == "fp64":
        knot, c = 70, int(counts[70])
        st = m.stencil(knot)
        pb = O.problem(O.PDE_TABLE, lut=fl, ulut=ul, vlut=vl, step=step)
        paths = O.simulate(pb, O.run_params(2e-3, 9, threads=8), m.x0[knot], m.y0[knot], st["rect"], knot, 0, c)
        o = O.reduce_batched(pb, paths, st, m.glob, [fac[min(max(int(v), 0), 3)] for v in st["kind"]], st["ipsi"],
                             32, 640, quirk=1)
        assert got["B"][knot] == o["B"] and got["BB"][knot] == o["BB"]
        assert np.array_equal(got["G"][m.row_ptr[knot]:m.row_ptr[knot + 1]], o["G"])
