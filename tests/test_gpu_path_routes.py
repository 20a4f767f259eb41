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
    """Paths per knot with which a launch takes the tiled kernel, if three of its tiles in four fit."""
    return int(eng.info()["n_cu"]) * 24 * 512 // int(np.sum(~mesh.on_boundary)) + 200


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


def _table(mode, n):
    """(samples, oracle dict, box) of the coefficient LUT of n x n samples."""
    from pdds_amd.workloads import varcoef_fields
    xs = np.linspace(-1, 1, n) if mode == 0 else -1 + (np.arange(n) + 0.5) * 2 / n
    X, Y = np.meshgrid(xs, xs)
    s = varcoef_fields(X, Y)
    return s, O.lut_dict(s, BOX, mode=mode)


def _knot_equals_oracle(got, mesh, olut, knot, n, h, seed):
    from pdds_amd.workloads import relative_fac
    fac = relative_fac(SW, NE, 4, 8, 1.0)
    st = mesh.stencil(knot)
    paths = O.simulate(O.problem(O.PDE_VARCOEF_LUT, lut=olut), O.run_params(h, seed, threads=8), mesh.x0[knot],
                       mesh.y0[knot], st["rect"], knot, 0, n)
    ref = O.reduce_batched(O.problem(O.PDE_VARCOEF_LUT, lut=olut), paths, st, mesh.glob,
                           [fac[min(max(int(v), 0), 3)] for v in st["kind"]], st["ipsi"], 32, 640, quirk=1)
    r = slice(mesh.row_ptr[knot], mesh.row_ptr[knot + 1])
    assert np.array_equal(got["G"][r], ref["G"]) and np.array_equal(got["Gvar"][r], ref["Gvar"])
    assert got["B"][knot] == ref["B"] and got["BB"][knot] == ref["BB"]


def _same(a, b, counters=("path_steps", "paths", "exits")):
    for k in ("G", "Gvar", "B", "BB"):
        assert np.array_equal(a[k], b[k]), k
    for k in counters:
        assert a["counters"][k] == b["counters"][k], k


# 96: every stencil's tile fits in LDS; 256: a segment's fits, a crossing's does not
@pytest.mark.parametrize("mode,n", [(0, 96), (0, 256), (1, 96)])
@pytest.mark.parametrize("precision", ["fp64", "fp32"])
def test_lut_assembly_is_the_same_in_every_kernel(eng, mesh, mode, n, precision):
    """Tiled with each row pitch, persistent, and the few-lanes kernel for part of the knots; FP64 also
    plain, and one knot of each the oracle's."""
    from pdds_amd.engine import bvp, default_run
    samples, olut = _table(mode, n)
    prob, many, h = bvp("varcoef_lut", lut=eng.lut(samples, BOX, mode=mode)), _many(eng, mesh), 4e-3
    counts = np.where(mesh.on_boundary, 0, many).astype(np.int64)
    counts[43] = 1500
    run = dict(h=h, seed=5, precision=precision, sub_batch=32, item_paths=640)
    print("lut", mode, n, precision, many, flush=True)
    ref = eng.assemble(mesh, prob, default_run(lut_lds=0, wg_size=128, **run), 0, paths_per_knot=counts)
    assert ref["counters"]["wg_size"] == 128
    for pad in (0, 1, 3, 7):
        got = eng.assemble(mesh, prob, default_run(lut_pad=pad, wg_size=128, **run), 0, paths_per_knot=counts)
        # (of 256 samples most tiles with 7 spare texels a row do not fit)
        assert got["counters"]["wg_size"] == (128 if pad == 7 and n == 256 and precision == "fp32" else TILED[precision]), pad
        _same(got, ref)
    few = np.where(np.arange(mesh.n_knots) == 42, 30011, np.where(np.arange(mesh.n_knots) == 43, 1500, 0))
    got = eng.assemble(mesh, prob, default_run(wg_size=128, **run), 0, paths_per_knot=few)
    assert got["counters"]["wg_size"] == 256
    ref2 = eng.assemble(mesh, prob, default_run(lut_lds=0, wg_size=128, **run), 0, paths_per_knot=np.where(few > 0, few, counts))
    assert ref2["counters"]["wg_size"] == 128
    for k in np.flatnonzero(few):
        r = slice(mesh.row_ptr[k], mesh.row_ptr[k + 1])
        assert np.array_equal(got["G"][r], ref2["G"][r]) and got["B"][k] == ref2["B"][k], k
    if precision == "fp64":
        _same(eng.assemble(mesh, prob, default_run(plain=1, **run), 0, paths_per_knot=counts), ref)
        _knot_equals_oracle(ref, mesh, olut, 43, 1500, h, 5)


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
def test_mixed_steps_are_the_same_in_every_kernel(eng, mesh, precision):
    """Knots of different step (adaptive h): every lane carries its knot's, in the tiled and in the
    persistent kernel; FP64 also the plain kernel's bits, and one knot the oracle's."""
    from pdds_amd.engine import bvp, default_run
    samples, olut = _table(0, 256)
    prob, many, h0 = bvp("varcoef_lut", lut=eng.lut(samples, BOX)), _many(eng, mesh), 0.02
    run = dict(h=h0, seed=11, precision=precision, adaptive_h=1, sub_batch=32, item_paths=640)
    hk = eng.knot_steps(mesh, prob, default_run(**run))
    knot = int(np.argmin(np.where(mesh.on_boundary, np.inf, hk)))
    assert 0 < hk[knot] < 0.75 * h0
    counts = np.where(mesh.on_boundary, 0, many).astype(np.int64)
    counts[knot] = 1100
    print("mixed", precision, many, "knot", knot, hk[knot], flush=True)
    got = eng.assemble(mesh, prob, default_run(**run), 0, paths_per_knot=counts)
    ref = eng.assemble(mesh, prob, default_run(lut_lds=0, wg_size=128, **run), 0, paths_per_knot=counts)
    assert got["counters"]["wg_size"] == TILED[precision] and ref["counters"]["wg_size"] == 128
    _same(got, ref)
    if precision == "fp64":
        _same(eng.assemble(mesh, prob, default_run(plain=1, **run), 0, paths_per_knot=counts), ref)
        _knot_equals_oracle(got, mesh, olut, knot, 1100, float(hk[knot]), 11)


def test_tiled_shards_are_bit_identical(eng, mesh):
    """Slices of the knots in launches of their own, each still tiled, put together give one
    assembly's bits."""
    from pdds_amd.engine import bvp, default_run
    samples, _ = _table(0, 256)
    prob, many = bvp("varcoef_lut", lut=eng.lut(samples, BOX)), 4 * _many(eng, mesh)
    run = default_run(h=8e-3, seed=29, sub_batch=32, item_paths=640)
    full = eng.assemble(mesh, prob, run, many)
    assert full["counters"]["wg_size"] == 512
    for shards in (2, 3):
        cuts = np.linspace(0, mesh.n_knots, shards + 1).astype(int)
        steps = 0
        for k0, k1 in zip(cuts[:-1], cuts[1:]):
            n = np.zeros(mesh.n_knots, dtype=np.int64)
            n[k0:k1] = many
            out = eng.assemble(mesh, prob, run, 0, paths_per_knot=n)
            print("shard", shards, k0, k1, out["counters"]["paths"], flush=True)
            r = slice(mesh.row_ptr[k0], mesh.row_ptr[k1])
            assert out["counters"]["wg_size"] == 512
            assert np.array_equal(out["G"][r], full["G"][r]) and np.array_equal(out["Gvar"][r], full["Gvar"][r])
            assert np.array_equal(out["B"][k0:k1], full["B"][k0:k1]) and np.array_equal(out["BB"][k0:k1], full["BB"][k0:k1])
            steps += out["counters"]["path_steps"]
        assert steps == full["counters"]["path_steps"]
