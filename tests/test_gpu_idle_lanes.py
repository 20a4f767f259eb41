"""Launches of a few paths of problems that read tables: lanes without a path take part in the reads,
and must change nothing.  Every kernel's sums are the plain kernel's, bit for bit (FP64)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
GLOB = np.array([-1.0, -1.0, 1.0, 1.0])


@pytest.fixture(scope="module")
def eng():
    from pdds_amd.engine import Engine
    e = Engine(0)
    yield e
    e.close()


@pytest.mark.parametrize("counts", [[1], [3], [17], [1, 1, 70], [2049]])
@pytest.mark.parametrize("kind,step", [("lut", 0), ("lut", 1), ("table", 0), ("table", 1), ("table", 2), ("table", 3)])
def test_few_paths_equal_plain(eng, kind, step, counts):
    from pdds_amd import workloads as W
    from pdds_amd.engine import bvp, default_run
    box = tuple(GLOB)
    if kind == "table":
        X, Y = np.meshgrid(np.linspace(-1, 1, 96), np.linspace(-1, 1, 96))
        prob = bvp("table", lut=eng.lut(W.varcoef_table_fields(X, Y), box), ulut=eng.lut(W.varcoef_u(X, Y), box),
                   vlut=eng.lut(W.varcoef_vrcv_fields(X, Y, 0.5), box))
    else:
        prob = bvp("varcoef_lut", lut=W.varcoef_lut(eng, 96, box))
    n = np.array(counts, dtype=np.int64)
    # the last point lies on the side of the square that the tables end at
    x, y = np.linspace(0.3, 0.999, len(n)), np.linspace(-0.2, 0.99, len(n))
    print(kind, step, counts, flush=True)
    ref = eng.point_eval(prob, default_run(h=2e-3, seed=7, step=step, plain=1), GLOB, x, y, n)
    for lds in (0, 1):
        got = eng.point_eval(prob, default_run(h=2e-3, seed=7, step=step, lut_lds=lds), GLOB, x, y, n)
        assert np.array_equal(got["u"], ref["u"]) and np.array_equal(got["u_var"], ref["u_var"])
        for k in ("path_steps", "exits"):
            assert got["counters"][k] == ref["counters"][k], k
