"""pdds_autotune times shapes of the kernel that large launches take, and only fields that it reads:
launches that do not differ are no candidates.  Results stay the base run's, bit for bit."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
SW, NE = (-1.0, -1.0), (1.0, 1.0)
BASE, TILED, UNTILED, FEW = 1, 4 * 2 * 4, 3 * 4 * 3, 4 * 3      # row pitch, grid, chunk; wg, grid, chunk; grid, chunk


@pytest.fixture(scope="module")
def eng():
    from pdds_amd.engine import Engine
    e = Engine(0)
    yield e
    e.close()


# problem, precision, step, candidates
CASES = [("helmholtz", "fp64", 0, BASE + FEW), ("helmholtz", "fp32", 0, BASE + FEW),
         ("helmholtz", "fp64", 1, BASE + UNTILED), ("monegros", "fp32", 0, BASE + UNTILED),
         ("varcoef", "fp64", 0, BASE + UNTILED), ("varcoef_lut", "fp32", 0, BASE + TILED + UNTILED),
         ("table", "fp64", 0, BASE + TILED + UNTILED), ("table", "fp64", 2, BASE + TILED + UNTILED),
         ("table", "fp32", 0, BASE + TILED + UNTILED), ("table", "fp32", 2, BASE + UNTILED)]


@pytest.mark.parametrize("pde,precision,step,candidates", CASES)
def test_candidates_differ_in_what_the_kernel_reads(eng, pde, precision, step, candidates):
    from pdds_amd.engine import Mesh, bvp, default_run
    from pdds_amd.workloads import relative_fac, table_problem, varcoef_lut
    m = Mesh(SW, NE, 4, 8, relative_fac(SW, NE, 4, 8, 1.0))
    pb = {"varcoef_lut": lambda: bvp(pde, lut=varcoef_lut(eng, 64, SW + NE)),
          "table": lambda: table_problem(eng, 64, SW + NE)}.get(pde, lambda: bvp(pde, k2=2.0))()
    base = default_run(h=4e-3, seed=3, precision=precision, step=step, wg_size=128, lut_pad=1)
    print(pde, precision, step, flush=True)
    best, rep = eng.autotune(m, pb, base, sample_paths=1024, max_knots=64, reps=1)
    assert rep["candidates"] == candidates and rep["best_rate"] >= rep["base_rate"] > 0
    if candidates == BASE + FEW:
        assert (best.wg_size, best.lut_lds, best.lut_pad) == (128, base.lut_lds, 1)
    a, b = eng.assemble(m, pb, base, 500), eng.assemble(m, pb, best, 500)
    for k in ("G", "Gvar", "B", "BB"):
        assert np.array_equal(a[k], b[k]), k
