"""Per-path records of problems that read tables: several lanes to a path up to a number of paths per
CU, one lane from there on (counters.wg_size: 256 and the run's own), with the same records on both
sides; and records of launches of many paths, whose waves take them in larger chunks."""
import numpy as np
import pytest

from oracle import oracle as O

pytestmark = pytest.mark.gpu
BOX = (-1.0, -1.0, 1.0, 1.0)
KEYS = ("steps", "xt", "yt", "Y", "Z", "xi")


@pytest.fixture(scope="module")
def eng():
    from pdds_amd.engine import Engine
    e = Engine(0)
    yield e
    e.close()


def _problem(eng, kind):
    from pdds_amd import workloads as W
    from pdds_amd.engine import bvp
    X, Y = np.meshgrid(np.linspace(-1, 1, 80), np.linspace(-1, 1, 80))
    if kind == "lut":
        s = W.varcoef_fields(X, Y)
        return bvp("varcoef_lut", lut=eng.lut(s, BOX)), O.problem(O.PDE_VARCOEF_LUT, lut=O.lut_dict(s, BOX))
    f, u = W.varcoef_table_fields(X, Y), W.varcoef_u(X, Y)
    return (bvp("table", lut=eng.lut(f, BOX), ulut=eng.lut(u, BOX)),
            O.problem(O.PDE_TABLE, lut=O.lut_dict(f, BOX), ulut=O.lut_dict(u, BOX)))


def _get(eng, prob, n, precision, phase2, h=2e-2):
    from pdds_amd.engine import default_run
    return eng.paths(prob, default_run(h=h, seed=5, precision=precision, wg_size=128), 0.1, -0.2, np.array(BOX), 4, 7, n,
                     phase2=phase2)


def _check_oracle(got, opb, n, phase2, h=2e-2):
    ref = O.simulate(opb, O.run_params(h, 5, phase2=int(phase2), threads=8), 0.1, -0.2, np.array(BOX), 4, 7, n,
                     **({"phase2_out": True} if phase2 else {}))
    for k in KEYS:
        assert np.array_equal(got[k][:n], ref[k]), k
        if phase2:
            assert np.array_equal(got["phase2"][k][:n], ref["phase2"][k]), ("phase2", k)


@pytest.mark.parametrize("kind,precision,phase2,most", [("lut", "fp64", False, 512), ("lut", "fp64", True, 1024),
                                                        ("lut", "fp32", False, 0), ("table", "fp64", False, 2048),
                                                        ("table", "fp64", True, 2048), ("table", "fp32", False, 256)])
def test_records_on_both_sides_of_the_limit(eng, kind, precision, phase2, most):
    prob, opb = _problem(eng, kind)
    n = most * eng.info()["n_cu"]
    print(kind, precision, phase2, n, flush=True)
    out = [_get(eng, prob, k, precision, phase2) for k in (n, n + 1) if k]
    assert [o["counters"]["wg_size"] for o in out] == [256, 128][2 - len(out):]
    if len(out) == 2:
        for k in KEYS:
            assert np.array_equal(out[0][k], out[1][k][:n]), k
            if phase2:
                assert np.array_equal(out[0]["phase2"][k], out[1]["phase2"][k][:n]), ("phase2", k)
    if precision == "fp64":
        _check_oracle(out[0], opb, 1500, phase2)


@pytest.mark.parametrize("n", [262144, 300007, 1000001])
@pytest.mark.parametrize("precision", ["fp64", "fp32"])
def test_records_of_many_paths(eng, n, precision):
    """The first and last thousand equal calls of their own."""
    from pdds_amd.engine import bvp, default_run
    print(n, precision, flush=True)
    prob, run = bvp("helmholtz", k2=2.0), default_run(h=2e-2, seed=5, precision=precision)
    got = eng.paths(prob, run, 0.1, -0.2, np.array(BOX), 4, 7, n)
    for first in (0, n - 1000):
        part = eng.paths(prob, run, 0.1, -0.2, np.array(BOX), 4, 7 + first, 1000)
        for k in KEYS:
            assert np.array_equal(got[k][first:first + 1000], part[k]), (first, k)
