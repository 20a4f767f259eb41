"""What pdds_point_eval_noalloc accepts and refuses near the end of its scratch array: a call is
counted by 32 bytes per path, 80 per work item, 208 per point and the small tables, each piece from a
256-byte boundary, whatever the descriptors that ride along take."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

DOMAIN = np.array([-1.0, -1.0, 1.0, 1.0])
SCRATCH = 64 << 20


@pytest.fixture(scope="module")
def eng():
    from pdds_amd.engine import Engine
    e = Engine(0)
    yield e
    e.close()


def _noalloc(eng, run, n_paths):
    from pdds_amd import _capi as A
    from pdds_amd.engine import bvp
    n = len(n_paths)
    x, y = np.linspace(-0.9, 0.9, n), np.linspace(0.8, -0.8, n)
    npth = np.ascontiguousarray(n_paths, dtype=np.int64)
    u, uv, ctr = np.full(n, np.nan), np.full(n, np.nan), A.Counters()
    st = A.lib().pdds_point_eval_noalloc(eng.h, C.byref(bvp("sinsin")._c()), C.byref(run), A.ptr(DOMAIN), n, A.ptr(x),
                                         A.ptr(y), A.ptr(npth, A._i64), A.ptr(u), A.ptr(uv), C.byref(ctr))
    return st, u, uv, x, y


def _counted(paths, items, points):
    """Bytes of the pieces in their order, each from a 256-byte boundary."""
    piece = [208, 256, 8, 8, 64, points * 96, items * 24, paths * 32, points * 16, items * 56, 8, points * 96, 64]
    end = 0
    for b in piece:
        end = -(-end // 256) * 256 + b
    return end


# one point whose every path is a work item, at the last number of paths that fits and the next; the
# most points that the estimate admits
@pytest.mark.parametrize("paths", ["last", "next", "spare"])
def test_many_work_items(eng, paths):
    from pdds_amd import _capi as A
    from pdds_amd.engine import bvp, default_run
    n = SCRATCH // 112
    while _counted(n, n, 1) > SCRATCH:
        n -= 1
    n = {"last": n - 64, "next": n + 64, "spare": n + 40000}[paths]
    run = default_run(h=2e-2, seed=31, sub_batch=1, item_paths=1)
    print("noalloc", paths, n, flush=True)
    st, u, uv, x, y = _noalloc(eng, run, [n])
    if paths != "last":
        assert st == A.ERR_FULL and b"64 MiB no-allocation scratch" in A.lib().pdds_last_error(eng.h)
        st, u, uv, x, y = _noalloc(eng, run, [2000])
        n = 2000
    assert st == A.OK
    ref = eng.point_eval(bvp("sinsin"), run, DOMAIN, x, y, np.array([n]))
    assert u[0] == ref["u"][0] and uv[0] == ref["u_var"][0]


@pytest.mark.parametrize("per_point", [1, 16])
def test_many_points(eng, per_point):
    from pdds_amd import _capi as A
    from pdds_amd.engine import bvp, default_run
    # 17 items a point in the estimate, and 65536 bytes of room
    points = (SCRATCH - 65536) // (32 * per_point + 208 + 17 * 80)
    run = default_run(h=2e-2, seed=31, sub_batch=1)
    print("noalloc", points, "points", flush=True)
    st, u, uv, x, y = _noalloc(eng, run, [per_point] * points)
    assert st == A.OK, A.lib().pdds_last_error(eng.h)
    ref = eng.point_eval(bvp("sinsin"), run, DOMAIN, x, y, np.full(points, per_point))
    assert np.array_equal(u, ref["u"]) and np.array_equal(uv, ref["u_var"], equal_nan=True)
    st = _noalloc(eng, run, [per_point] * (points + 1))[0]
    assert st == A.ERR_FULL
