"""The group path kernel (1, 4 or 16 lanes to a path) against the plain kernel, one lane to a path
from start to end: point estimates, variances, step counts and exits equal bit for bit, FP64 and
FP32, for path counts on both sides of every change of the group's width, for launches whose last
waves and groups are partly filled, for ragged counts over several knots and with a step cap that
falls inside a group's steps."""
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


def _both(eng, problem, counts, **run):
    from pdds_amd.engine import default_run
    n = len(counts)
    x = np.linspace(-0.9, 0.8, n)
    y = np.linspace(0.7, -0.6, n)
    return [eng.point_eval(problem, default_run(plain=plain, **run), GLOB, x, y, counts) for plain in (0, 1)]


def _equal(a, b):
    assert np.array_equal(a["u"], b["u"]) and np.array_equal(a["u_var"], b["u_var"])
    for k in ("path_steps", "paths", "exits", "capped"):
        assert a["counters"][k] == b["counters"][k], k


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("total", ["one", "ragged-16", "last-16", "first-4", "last-4", "first-1"])
def test_group_widths_equal_plain(eng, precision, total):
    from pdds_amd.engine import bvp
    cu = eng.info()["n_cu"]
    one_lane = cu * (4096 if precision == "fp64" else 2048)
    counts = {"one": [1], "ragged-16": [17, 1, 333, 64, 5], "last-16": [cu * 32], "first-4": [cu * 32 - 6, 7],
              "last-4": [one_lane - 4, 3], "first-1": [one_lane - 3, 3]}[total]
    print(precision, total, counts, flush=True)
    # a step large enough that the longest of a million paths stays short
    _equal(*_both(eng, bvp("helmholtz", k2=3.0), np.array(counts), h=0.01, seed=5, precision=precision))


@pytest.mark.parametrize("pde", ["sinsin", "monegros"])
def test_group_problems_equal_plain(eng, pde):
    from pdds_amd.engine import bvp
    print(pde, flush=True)
    _equal(*_both(eng, bvp(pde), np.array([3000, 1, 40, 9001]), h=0.004, seed=9))


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
def test_group_widths_equal_each_other(eng, precision):
    """The same points alone (16 lanes), beside one that takes the launch to 4 lanes and beside one
    that takes it to 1.  (The plain FP32 kernel of this problem rounds differently.)"""
    from pdds_amd.engine import bvp, default_run
    cu = eng.info()["n_cu"]
    x, y, n = np.array([0.1, -0.6, 0.4]), np.array([-0.3, 0.2, 0.9]), np.array([3000, 41, 700])
    out = []
    for extra in (0, cu * 32, cu * 4096):
        print(precision, extra, flush=True)
        m = 3 + (extra > 0)
        r = eng.point_eval(bvp("sinsin"), default_run(h=0.01, seed=9, precision=precision), GLOB, np.append(x, 0.5)[:m],
                           np.append(y, 0.5)[:m], np.append(n, extra)[:m])
        out.append((r["u"][:3], r["u_var"][:3]))
    for u, v in out[1:]:
        assert np.array_equal(u, out[0][0]) and np.array_equal(v, out[0][1])


@pytest.mark.parametrize("case", ["varcoef", "varcoef_lut", "table", "helmholtz-robin", "varcoef-robin"])
@pytest.mark.parametrize("precision", ["fp64", "fp32"])
def test_group_equals_one_lane_kernels(eng, case, precision):
    """Problems whose coefficients move the path, and reflecting sides: the same points in a launch
    small enough for the group kernel and in one that the other path kernels take."""
    from pdds_amd.engine import bvp, default_run
    from pdds_amd.workloads import table_problem, varcoef_lut
    if case.endswith("robin") and precision == "fp32":
        pytest.skip("FP32 reflecting launches have no group form")
    pb = {"varcoef": lambda: bvp("varcoef"), "varcoef_lut": lambda: bvp("varcoef_lut", lut=varcoef_lut(eng, 64)),
          "table": lambda: table_problem(eng, 64), "helmholtz-robin": lambda: bvp("helmholtz", k2=2.0, neumann=10, varphi=-1.0),
          "varcoef-robin": lambda: bvp("varcoef", neumann=1, varphi=-0.5, rho=0.2)}[case]()
    cu = eng.info()["n_cu"]
    x, y, n = np.array([0.1, -0.6, 0.4]), np.array([-0.3, 0.2, 0.9]), np.array([3000, 41, 700])
    out = []
    for extra in (0, cu * 2048 - int(n.sum()), cu * 2048):
        print(case, precision, extra, flush=True)
        m = 3 + (extra > 0)
        r = eng.point_eval(pb, default_run(h=0.01, seed=9, precision=precision), GLOB, np.append(x, 0.5)[:m],
                           np.append(y, 0.5)[:m], np.append(n, extra)[:m])
        out.append((r["u"][:3], r["u_var"][:3]))
    for u, v in out[1:]:
        assert np.array_equal(u, out[0][0]) and np.array_equal(v, out[0][1])


@pytest.mark.parametrize("n,path0,cap", [(1, 0, 0), (63, 5, 0), (1000, (1 << 32) - 1000, 0), (700, 0, 7)])
@pytest.mark.parametrize("refl", [0, 8])
def test_group_records_equal_oracle(eng, n, path0, cap, refl):
    """pdds_paths: partly filled waves, the last path numbers, a cap within the first and the second
    phase's steps; both phases equal the oracle's records."""
    from oracle import oracle as O
    from pdds_amd.engine import bvp, default_run
    rect = np.array([-0.6, -0.9, 0.4, 0.2])
    print(n, path0, cap, refl, flush=True)
    got = eng.paths(bvp("helmholtz", k2=2.0, neumann=refl), default_run(h=4e-3, seed=7, max_steps=cap), 0.1, -0.2, rect, 5,
                    path0, n, phase2=True)
    run = O.run_params(4e-3, 7, phase2=1, threads=8)
    if cap:
        run.max_steps = cap
    ref = O.simulate(O.problem(O.PDE_HELMHOLTZ, k2=2.0, refl=refl), run, 0.1, -0.2, rect, 5, path0, n, phase2_out=True)
    for k in ("steps", "xt", "yt", "Y", "Z", "xi"):
        assert np.array_equal(got[k], ref[k]), k
        assert np.array_equal(got["phase2"][k], ref["phase2"][k]), ("phase2", k)


@pytest.mark.parametrize("cap", [1, 2, 15, 16, 17, 33])
@pytest.mark.parametrize("precision", ["fp64", "fp32"])
def test_group_step_cap_equals_plain(eng, precision, cap):
    from pdds_amd.engine import bvp
    print(precision, "cap", cap, flush=True)
    a, b = _both(eng, bvp("helmholtz", k2=2.0), np.array([500, 77]), h=0.002, seed=3, precision=precision, max_steps=cap)
    assert a["counters"]["capped"] > 0
    _equal(a, b)


def test_group_mixed_launch_equals_plain(eng):
    """Knots of different step (adaptive h) in one launch: every group carries its knot's."""
    from pdds_amd.engine import Mesh, bvp, default_run
    from pdds_amd.workloads import relative_fac
    m = Mesh((-1.0, -1.0), (1.0, 1.0), 3, 9, relative_fac((-1.0, -1.0), (1.0, 1.0), 3, 9, 1.0))
    n = np.random.default_rng(2).integers(1, 900, m.n_knots)
    for precision in ("fp64", "fp32"):
        a, b = (eng.assemble(m, bvp("helmholtz", k2=4.0),
                             default_run(h=0.02, seed=4, adaptive_h=1, precision=precision, plain=plain), 0,
                             paths_per_knot=n) for plain in (0, 1))
        for k in ("G", "Gvar", "B", "BB"):
            assert np.array_equal(a[k], b[k], equal_nan=True), (precision, k)
        assert a["counters"]["path_steps"] == b["counters"]["path_steps"]
