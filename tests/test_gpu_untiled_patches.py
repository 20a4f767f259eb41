"""Tiled launches in which some or all stencils' tiles do not fit in LDS: their patch reads its tables
from global memory, also on a pass whose last paths stop in its first step (the FP32 kernels of
two steps a pass).  Results are those of the persistent kernel, bit for bit."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
SW, NE = (-1.0, -1.0), (1.0, 1.0)


@pytest.fixture(scope="module")
def eng():
    from pdds_amd.engine import Engine
    e = Engine(0)
    yield e
    e.close()


def _equal(eng, mesh, problem, counts, wg, **run):
    from pdds_amd.engine import default_run
    a, b = (eng.assemble(mesh, problem, default_run(lut_lds=lds, wg_size=128, **run), 0, paths_per_knot=counts) for lds in (1, 0))
    assert a["counters"]["wg_size"] == wg and b["counters"]["wg_size"] == 128
    for k in ("G", "Gvar", "B", "BB"):
        assert np.array_equal(a[k], b[k]), k
    for k in ("path_steps", "exits", "paths"):
        assert a["counters"][k] == b["counters"][k], k


@pytest.mark.parametrize("precision", ["fp32", "fp64"])
def test_table_with_some_tiles(eng, precision):
    from pdds_amd.engine import Mesh
    from pdds_amd.workloads import relative_fac, table_problem
    # the crossing's stencil does not fit, the others' do: 4.3 10^6 paths
    m = Mesh(SW, NE, 4, 16, relative_fac(SW, NE, 4, 16, 0.8))
    counts = np.where(m.on_boundary, 0, 12500).astype(np.int64)
    counts[70] = 5437
    print("table 160", precision, flush=True)
    _equal(eng, m, table_problem(eng, 160, SW + NE), counts, 512, h=8e-3, seed=9, precision=precision)


# 1024: a sector's box covers at least 150 x 150 texels of 16 bytes, no tile fits; 256: a fifth do not
@pytest.mark.parametrize("precision,n", [("fp64", 1024), ("fp64", 256), ("fp32", 256)])
def test_disc_without_tiles(eng, precision, n):
    from pdds_amd.engine import Mesh, bvp
    from pdds_amd.workloads import varcoef_lut
    m = Mesh.disc(1.0, 3, 8, 11, 6, 12, 1.0)
    counts = np.where(m.on_boundary, 0, 8000).astype(np.int64)
    counts[5] = 321
    print("disc", n, precision, flush=True)
    _equal(eng, m, bvp("varcoef_lut", lut=varcoef_lut(eng, n, SW + NE)), counts, 512, h=1e-3, seed=4, precision=precision)
