"""Which path kernel a launch takes, as counters.wg_size tells it -- 256 threads: several lanes to a
path; 512 (FP64) or 768 (FP32): LDS-tiled; the run's own wg_size: persistent or plain -- and that
each of them gives the same bits."""
import numpy as np
import pytest

from oracle import oracle as O

pytestmark = pytest.mark.gpu
SW, NE = (-1.0, -1.0), (1.0, 1.0)
BOX = SW + NE
TILED = {"fp64": 512, "fp32": 768}


@pytest.fixture(scope="module")
def eng():
    from pdds_amd.engine import Engine
    e = Engine(0)
    yield e
    e.close()


@pytest.fixture(scope="module")
def mesh():
    from pdds_amd.engine import Mesh
    from pdds_amd.workloads import relative_fac
    return Mesh(SW, NE, 4, 8, relative_fac(SW, NE, 4, 8, 1.0))


def _many(eng, mesh):
    """Paths per knot with which a launch has more than 2048 paths per CU."""
    return int(eng.info()["n_cu"]) * 2048 // int(np.sum(~mesh.on_boundary)) + 200


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
def test_counters_report_the_launched_work_group(eng, mesh, precision):
    from pdds_amd.engine import bvp, default_run
    from pdds_amd.workloads import varcoef_lut
    prob, many = bvp("varcoef_lut", lut=varcoef_lut(eng, 64, BOX)), _many(eng, mesh)

    def wg(n, **run):
        print(precision, n, run, flush=True)
        return eng.assemble(mesh, prob, default_run(h=1e-2, seed=3, precision=precision, **run), n)["counters"]["wg_size"]

    assert wg(100) == 256 and wg(100, wg_size=64) == 256 and wg(100, wg_size=64, lut_lds=0) == 256
    assert wg(100, wg_size=64, plain=1) == 64
    assert wg(many) == TILED[precision] and wg(many, wg_size=64) == TILED[precision]
    assert wg(many, wg_size=128, lut_lds=0) == 128
