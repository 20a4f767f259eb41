"""The reflected step at a corner of two reflecting sides, whose normal has two components: per-path
records (4 lanes to a path) and point estimates (16 and 4 lanes, one lane, plain kernel) equal to
the oracle's, bit for bit.  A path comes to step from a corner where it starts past one, and where
its projection back onto the corner rounds outwards in both coordinates, as it does at the
south-west corner of the boxes here."""
import numpy as np
import pytest

from oracle import oracle as O

pytestmark = pytest.mark.gpu

# N 1, S 2, E 4, W 8
CORNERS = {"NE": (5, 1, 1), "SE": (6, 1, -1), "NW": (9, -1, 1), "SW": (10, -1, -1)}
BOXES = {"a": (-3.96, -3.96, -1.97, -1.97), "b": (-5.0, -5.0, -1.1, -1.1), "c": (-1.0, -1.0, -0.2, -0.2)}
PDES = {"sinsin": O.PDE_SINSIN, "helmholtz": O.PDE_HELMHOLTZ, "monegros": O.PDE_MONEGROS, "varcoef": O.PDE_VARCOEF}


@pytest.fixture(scope="module")
def eng():
    from pdds_amd.engine import Engine
    e = Engine(0)
    yield e
    e.close()


def _at(box, corner, frac):
    """The point frac of the width outside the corner along x, and 0.8 frac along y (inside: frac < 0)."""
    _, sx, sy = CORNERS[corner]
    w = box[2] - box[0]
    return ((box[2] if sx > 0 else box[0]) + sx * frac * w, (box[3] if sy > 0 else box[1]) + sy * 0.8 * frac * w)


def _rounds_outwards(box):
    b = np.array(box)
    c = 0.5 * (b[:2] + b[2:])
    h = b[2:] - c
    return bool(np.all(c - (c - h) > h))


def _records(eng, pde, box, corner, rho, frac, n):
    from pdds_amd.engine import bvp, default_run
    mask = CORNERS[corner][0]
    h = (0.03 * (box[2] - box[0])) ** 2
    x0, y0 = _at(box, corner, frac)
    print("corner records", pde, box, corner, "rho", rho, "x0", (x0, y0), flush=True)
    got = eng.paths(bvp(pde, k2=2.0, neumann=mask, varphi=-1.0, rho=rho), default_run(h=h, seed=7), x0, y0,
                    np.array(box), 5, 0, n, phase2=True)
    ref = O.simulate(O.problem(PDES[pde], k2=2.0, refl=mask, robin=-1.0, rho=rho),
                     O.run_params(h, 7, phase2=1, threads=8), x0, y0, np.array(box), 5, 0, n, phase2_out=True)
    for k in ("steps", "xt", "yt", "Y", "Z", "xi"):
        assert np.array_equal(got[k], ref[k]), (k, int(np.sum(got[k] != ref[k])))
        assert np.array_equal(got["phase2"][k], ref["phase2"][k]), ("phase2", k)


@pytest.mark.parametrize("pde", list(PDES))
@pytest.mark.parametrize("corner", list(CORNERS))
@pytest.mark.parametrize("rho", [0.0, 1e-3])
def test_records_from_past_a_corner(eng, pde, corner, rho):
    # (with a band of local time a start outside it steps from the corner all the same: d > 0)
    _records(eng, pde, BOXES["c"], corner, rho, 0.02, 300)


@pytest.mark.parametrize("pde", ["sinsin", "helmholtz", "monegros"])
@pytest.mark.parametrize("box", list(BOXES))
@pytest.mark.parametrize("rho", [0.0, 1e-3, 0.05])
def test_records_projected_onto_a_corner(eng, pde, box, rho):
    assert _rounds_outwards(BOXES[box])
    _records(eng, pde, BOXES[box], "SW", rho, -0.1, 1000)


@pytest.mark.parametrize("box", list(BOXES))
@pytest.mark.parametrize("rho", [0.0, 1e-3, 0.05])
def test_points_near_a_corner(eng, box, rho):
    """The same two points alone (16 lanes), beside one that takes the launch to 4 lanes and beside
    one that takes it to the kernel of one lane; and in the plain kernel."""
    from pdds_amd.engine import bvp, default_run
    glob = np.array(BOXES[box])
    h = (0.03 * (glob[2] - glob[0])) ** 2
    cu = eng.info()["n_cu"]
    p = [_at(glob, "SW", f) for f in (-0.1, -0.05, -0.7)]
    x, y = np.array([q[0] for q in p]), np.array([q[1] for q in p])
    pb = O.problem(O.PDE_SINSIN, refl=10, robin=-1.0, rho=rho)
    st = {"rect": glob, "msz": np.zeros(4, dtype=np.int32), "idx": np.zeros(0, dtype=np.int32),
          "px": np.zeros(0), "py": np.zeros(0)}
    want = []
    for i in range(2):
        paths = O.simulate(pb, O.run_params(h, 5, threads=8), x[i], y[i], glob, i, 0, 2000)
        want.append(O.reduce_batched(pb, paths, st, glob, [1.0] * 4, [np.zeros((0, 0))] * 4, 32, 512)["B"])
    for extra, plain in ((0, 0), (cu * 32, 0), (cu * 2048, 0), (0, 1)):
        m = 3 if extra else 2
        print("corner points", box, rho, extra, plain, flush=True)
        got = eng.point_eval(bvp("sinsin", neumann=10, varphi=-1.0, rho=rho),
                             default_run(h=h, seed=5, item_paths=512, plain=plain), glob, x[:m], y[:m],
                             np.array([2000, 2000, extra])[:m])
        assert got["u"][0] == want[0] and got["u"][1] == want[1], (extra, plain)
