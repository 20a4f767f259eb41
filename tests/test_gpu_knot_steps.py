"""Step and step-cap sums of the persistent and tiled path kernels (one lane to a path), which a wave holds for
the knots its pool came to last: knots of one path, of fewer than a wave takes at once and of
many, one after another in one launch; a step cap that stops some paths.  Sums and results are
the plain kernel's."""
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


def _counts(kind):
    rng = np.random.default_rng(5)
    return {"ones": np.ones(700, dtype=np.int64),
            "few": rng.integers(1, 9, 3000),
            "mixed": np.where(rng.random(400) < 0.7, rng.integers(1, 70, 400), rng.integers(2000, 4000, 400)),
            "one": np.array([150001], dtype=np.int64)}[kind].astype(np.int64)


@pytest.mark.parametrize("kind", ["ones", "few", "mixed", "one"])
# (forms without several lanes to a path: the plain step, and FP32 paths with a reflecting side)
@pytest.mark.parametrize("precision,pde,step,neumann,cap", [("fp64", "helmholtz", 1, 0, 0), ("fp32", "helmholtz", 1, 0, 0),
                                                            ("fp64", "varcoef", 1, 0, 30), ("fp32", "varcoef", 1, 0, 30),
                                                            ("fp32", "monegros", 1, 0, 0), ("fp32", "helmholtz", 0, 8, 0),
                                                            ("fp64", "varcoef_lut", 1, 0, 0), ("fp32", "varcoef_lut", 1, 0, 25),
                                                            ("fp64", "table", 1, 0, 25), ("fp64", "table", 2, 0, 0)])
def test_step_sums_equal_plain(eng, kind, precision, pde, step, neumann, cap):
    from pdds_amd.engine import bvp, default_run
    n = _counts(kind)
    x, y = np.linspace(-0.9, 0.8, len(n)), np.linspace(0.7, -0.6, len(n))
    from pdds_amd.workloads import table_problem, varcoef_lut
    prob = {"varcoef_lut": lambda: bvp(pde, lut=varcoef_lut(eng, 64, tuple(GLOB))),
            "table": lambda: table_problem(eng, 64, tuple(GLOB))}.get(pde, lambda: bvp(pde, neumann=neumann))()
    run = dict(h=5e-3, seed=3, precision=precision, wg_size=128, step=step, max_steps=cap)
    print(kind, precision, pde, step, neumann, cap, flush=True)
    a, b = (eng.point_eval(prob, default_run(plain=p, **run), GLOB, x, y, n) for p in (0, 1))
    assert a["counters"]["wg_size"] == 128
    for k in ("path_steps", "paths", "exits", "capped"):
        assert a["counters"][k] == b["counters"][k], k
    assert np.array_equal(a["u"], b["u"]) and np.array_equal(a["u_var"], b["u_var"])
    assert (a["counters"]["capped"] > 0) == (cap > 0)


@pytest.mark.parametrize("kind", ["ones", "mixed", "one"])
@pytest.mark.parametrize("cap", [0, 25])
def test_tiled_step_sums_equal_persistent(eng, kind, cap):
    """The tiled kernel's FP32 sums, for the two knots a wave came to last."""
    from pdds_amd.engine import bvp, default_run
    from pdds_amd.workloads import varcoef_lut
    # above four paths a lane of the tiled grid
    extra = eng.info()["n_cu"] * 768 * 4
    n = np.append(_counts(kind), [extra // 3, 7, extra])
    x, y = np.linspace(-0.9, 0.8, len(n)), np.linspace(0.7, -0.6, len(n))
    prob = bvp("varcoef_lut", lut=varcoef_lut(eng, 64, tuple(GLOB)))
    print(kind, cap, flush=True)
    a, b = (eng.point_eval(prob, default_run(h=1e-2, seed=3, precision="fp32", wg_size=128, lut_lds=lds, max_steps=cap),
                           GLOB, x, y, n) for lds in (1, 0))
    assert a["counters"]["wg_size"] == 768 and b["counters"]["wg_size"] == 128
    for k in ("path_steps", "paths", "exits", "capped"):
        assert a["counters"][k] == b["counters"][k], k
    assert np.array_equal(a["u"], b["u"]) and np.array_equal(a["u_var"], b["u_var"])
    assert (a["counters"]["capped"] > 0) == (cap > 0)
