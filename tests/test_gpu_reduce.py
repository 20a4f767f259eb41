"""The reduction's work-groups against the oracle: groups of 16 sub-batches on the matrix units
(stencils of up to 16 tiles of 16 side entries, of up to 32), the kernel for what they do not take,
sub-batch sizes that divide 64 and that do not, spans of several items and groups that end inside an
item.  G, its variance, B, BB and the equation sums are the oracle's bits."""
import numpy as np
import pytest

from oracle import oracle as O

pytestmark = pytest.mark.gpu
BOX = ((-1.0, -1.0), (1.0, 1.0))


@pytest.fixture(scope="module")
def eng():
    from pdds_amd.engine import Engine
    e = Engine(0)
    yield e
    e.close()


def _tiles(m):
    return np.array([sum((int(v) + 15) // 16 for v in m.stencil(k)["msz"]) for k in range(m.n_knots)])


def _mesh(n_sub, n_node):
    from pdds_amd.engine import Mesh
    from pdds_amd.workloads import relative_fac
    fac = relative_fac(BOX[0], BOX[1], n_sub, n_node, 0.8)
    return Mesh(BOX[0], BOX[1], n_sub, n_node, fac), fac


def _check(got, k, m, fac, quirk, S, P, n, h, seed, u=None):
    st = m.stencil(k)
    paths = O.simulate(O.problem(O.PDE_SINSIN), O.run_params(h, seed, threads=8), m.x0[k], m.y0[k], st["rect"], k, 0, n)
    cs = [fac[min(max(int(v), 0), 3)] for v in st["kind"]]
    ref = O.reduce_batched_eq(O.problem(O.PDE_SINSIN), paths, st, m.glob, cs, st["ipsi"], S, P,
                              np.zeros(m.n_knots) if u is None else u, quirk=quirk)
    r = slice(m.row_ptr[k], m.row_ptr[k + 1])
    order = np.argsort(ref["cols"], kind="stable")
    assert np.array_equal(m.cols[r][np.argsort(m.cols[r], kind="stable")], ref["cols"][order])
    mine = np.argsort(m.cols[r], kind="stable")
    assert np.array_equal(got["G"][r][mine], ref["G"][order]), (k, S)
    assert np.array_equal(got["Gvar"][r][mine], ref["Gvar"][order]), (k, S)
    assert got["B"][k] == ref["B"] and got["BB"][k] == ref["BB"], (k, S)
    if u is not None:
        assert got["eq_mean"][k] == ref["eq_mean"] and got["eq_var"][k] == ref["eq_var"], (k, S)


# nodes per interface: 8 (few tiles), 30 (up to 16 and more), 70 (more than 32 tiles for some)
@pytest.mark.parametrize("quirk", [1, 0])
@pytest.mark.parametrize("n_node,S,n", [(8, 32, 1700), (8, 16, 1501), (8, 64, 2500), (8, 1, 40), (8, 48, 1000),
                                        (8, 100, 3333), (8, 300, 2000), (30, 32, 1650), (30, 64, 3000), (70, 32, 1000)])
def test_assembly_matches_the_oracle(eng, n_node, S, n, quirk):
    from pdds_amd.engine import bvp, default_run
    m, fac = _mesh(4, n_node)
    tiles = _tiles(m)
    h, seed = 1e-3, 31
    rng = np.random.default_rng(S)
    counts = rng.integers(n // 2, n + 1, m.n_knots)
    counts[::7] = rng.integers(1, 4, len(counts[::7])) * S
    run = default_run(h=h, seed=seed, quirk_last_side=quirk, sub_batch=S)
    u = np.cos(3 * m.px) * np.cos(2 * m.py) if quirk == 0 else None
    if u is None:
        got = eng.assemble(m, bvp("sinsin"), run, n, paths_per_knot=counts)
    else:
        got = eng.assemble_eq(m, bvp("sinsin"), run, n, u, paths_per_knot=counts)
    mc = np.flatnonzero(~m.on_boundary)
    some = {int(mc[np.argmin(tiles[mc])]), int(mc[np.argmax(tiles[mc])]), int(mc[len(mc) // 2]), int(mc[0]),
            int(mc[mc % 7 == 0][0])}
    for k in sorted(some):
        c = int(counts[k])
        q = max(1, (c + 16 * S - 1) // (16 * S))
        _check(got, k, m, fac, quirk, S, q * S, c, h, seed, u)


def test_spans_and_long_items_match_the_oracle(eng):
    """Items of 40 sub-batches (groups that end inside an item) and of one (16 to a group)."""
    from pdds_amd.engine import bvp, default_run
    m, fac = _mesh(8, 8)
    for P in (32, 64, 1280):
        run = default_run(h=2e-3, seed=5, sub_batch=32, item_paths=P)
        got = eng.assemble(m, bvp("sinsin"), run, 2600)
        for k in np.flatnonzero(~m.on_boundary)[[3, 200, 401]]:
            _check(got, int(k), m, fac, 1, 32, P, 2600, 2e-3, 5)
