"""The reduction with and without the sums of the knot equations, at stencils and sub-batches on both
sides of the limit between its two kernels: each entry's Gaussian values are formed by two codes of
the exponential, which give the same bits."""
import numpy as np
import pytest

from oracle import oracle as O

pytestmark = pytest.mark.gpu
SW, NE = (-1.0, -1.0), (1.0, 1.0)


@pytest.fixture(scope="module")
def eng():
    from pdds_amd.engine import Engine
    e = Engine(0)
    yield e
    e.close()


# sides of 8 knots (16 side entries fit the first kernel, sub-batches of 100 do not), of 70 (neither)
@pytest.mark.parametrize("n_node,fac,sub_batch", [(8, 0.8, 32), (8, 0.8, 100), (70, 0.6, 32), (70, 0.6, 100), (70, 0.1, 48)])
@pytest.mark.parametrize("precision", ["fp64", "fp32"])
def test_plain_and_equation_sums_agree(eng, n_node, fac, sub_batch, precision):
    from pdds_amd.engine import Mesh, bvp, default_run
    from pdds_amd.workloads import relative_fac
    f = relative_fac(SW, NE, 4, n_node, fac)
    m = Mesh(SW, NE, 4, n_node, f)
    counts = np.where(m.on_boundary, 0, 300).astype(np.int64)
    knot = int(np.flatnonzero(~m.on_boundary)[5])
    counts[knot] = 1237
    run = default_run(h=8e-3, seed=5, precision=precision, sub_batch=sub_batch, item_paths=20 * sub_batch)
    prob = bvp("helmholtz", k2=3.0)
    print(n_node, fac, sub_batch, precision, flush=True)
    a = eng.assemble(m, prob, run, 0, paths_per_knot=counts)
    b = eng.assemble_eq(m, prob, run, 0, np.cos(m.px), paths_per_knot=counts)
    for k in ("G", "Gvar", "B", "BB"):
        assert np.array_equal(a[k], b[k]), k
    if precision == "fp64":
        st, pb = m.stencil(knot), O.problem(O.PDE_HELMHOLTZ, k2=3.0)
        paths = O.simulate(pb, O.run_params(8e-3, 5, threads=8), m.x0[knot], m.y0[knot], st["rect"], knot, 0, 1237)
        o = O.reduce_batched(pb, paths, st, m.glob, [f[min(max(int(v), 0), 3)] for v in st["kind"]], st["ipsi"],
                             sub_batch, 20 * sub_batch, quirk=1)
        r = slice(m.row_ptr[knot], m.row_ptr[knot + 1])
        assert a["B"][knot] == o["B"] and a["BB"][knot] == o["BB"] and np.array_equal(a["G"][r], o["G"])
