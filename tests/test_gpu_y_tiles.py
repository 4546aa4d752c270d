"""The Y sweep's LDS tiles (16 columns x 32 rows; domains of up to a few million cells) against the
oracle and against the marching runs that larger domains take (`y_run_rows` set), bit for bit, at the
edges of the tiles, with both ways of making the time step: in the cycle's first sweep (tiles, two
or three sweeps a cycle) and by a kernel of its own (marches, single-sweep splittings). The batch
likewise: its default and its marches."""
import numpy as np
import pytest

FIELDS = ("rho", "umat", "vmat", "Emat", "pmat", "cmat")
GAD2 = dict(scheme=1, projection=2, limiter=1, nb_ghosts=4)
GOD1 = dict(scheme=0, projection=1, nb_ghosts=2)
GAD1 = dict(scheme=1, projection=1, limiter=2, nb_ghosts=5)
GOD2 = dict(scheme=0, projection=2, nb_ghosts=3)


def _run(armon, test, **kw):
    r, s = armon.run(armon.make_params(test, verbose=5, **kw))
    assert r.status == 0, armon.errors()
    out = {f: s.read(f) for f in FIELDS}, r.cycles, r.final_dt
    s.close()
    return out


# GAD + second order writes 24 rows of a tile's 32, Godunov + first order 28, the others 26
@pytest.mark.gpu
@pytest.mark.parametrize("nx,ny,scheme,splitting", [
    (15, 24, GAD2, 0), (16, 25, GAD2, 1), (17, 23, GAD2, 2), (33, 49, GAD2, 4), (4, 4, GAD2, 1), (64, 8, GAD2, 3),
    (16, 28, GOD1, 0), (31, 29, GOD1, 2), (5, 57, GOD1, 1), (16, 26, GAD1, 1), (47, 27, GAD1, 0), (32, 53, GOD2, 2)])
def test_tiles_are_the_oracle(armon, po, oracle, nx, ny, scheme, splitting):
    kw = dict(nx=nx, ny=ny, axis_splitting=splitting, max_cycles=9, cfl=0.5, **scheme)
    got, cycles, dt = _run(armon, "Sod_circ", **kw)
    march, _, _ = _run(armon, "Sod_circ", y_run_rows=7, **kw)
    op = po.make_params(oracle, "Sod_circ", verbose=5, **kw)
    status, data, ocycles, odt, _ = po.run(oracle, op)
    assert status == 0 and (cycles, dt) == (ocycles, odt)
    mask = data.array("domain_mask") == 1
    for f in FIELDS:
        assert np.array_equal(got[f][mask], data.array(f)[mask]), f
        assert np.array_equal(got[f], march[f]), f


@pytest.mark.gpu
@pytest.mark.parametrize("test,nx,ny", [("Sedov", 50, 75), ("Bizarrium", 33, 25), ("Sod", 129, 24)])
def test_fp32_tiles_are_the_marches(armon, test, nx, ny):
    kw = dict(nx=nx, ny=ny, axis_splitting=1, max_cycles=12, precision=armon.PREC_FP32_MIXED, **GAD2)
    (a, ca, da), (b, cb, db) = _run(armon, test, **kw), _run(armon, test, y_run_rows=9, **kw)
    assert (ca, da) == (cb, db)
    for f in FIELDS:
        assert np.array_equal(a[f], b[f]), f


# the smallest domain above the tiles' limit marches, the largest below it does not
@pytest.mark.gpu
@pytest.mark.parametrize("ny", [2560, 2561])
def test_the_rule_on_the_number_of_cells(armon, ny):
    kw = dict(nx=1024, ny=ny, max_cycles=3, **GAD2)
    (a, _, da), (b, _, db) = _run(armon, "Sedov", **kw), _run(armon, "Sedov", y_run_rows=64, **kw)
    assert da == db
    for f in FIELDS:
        assert np.array_equal(a[f], b[f]), f


# the largest domain whose first sweep makes the time step and the smallest one with a launch for it
@pytest.mark.gpu
@pytest.mark.parametrize("precision,ny", [(0, 896), (0, 897), (1, 2048), (1, 2049)])
def test_the_rule_on_the_time_step(armon, precision, ny):
    kw = dict(nx=1024, ny=ny, max_cycles=4, precision=precision, axis_splitting=1, **GAD2)
    (a, _, da), (b, _, db) = _run(armon, "Sedov", **kw), _run(armon, "Sedov", y_run_rows=64, **kw)
    assert da == db
    for f in FIELDS:
        assert np.array_equal(a[f], b[f]), f


@pytest.mark.gpu
@pytest.mark.parametrize("precision,splitting,rows", [(0, 0, 16), (0, 2, 33), (1, 1, 64), (0, 4, 5)])
def test_batch_tiles_are_its_marches(armon, precision, splitting, rows):
    def run(march):
        common = armon.batch_params(max_cycles=11, axis_splitting=splitting, precision=precision, verbose=5, cfl=0.6,
                                    **GAD2)
        b = armon.Batch(common, armon.random_specs(31, 9, 24 * 24, 96 * 96))
        if march:
            b.set_tuning(rows)
        b.init()
        b.begin()
        b.run()
        assert b.finish() == 0, armon.errors()
        out = [(b.result(d).cycles, b.result(d).final_dt, [b.read(d, f) for f in FIELDS]) for d in range(b.n)]
        b.close()
        return out

    for (ca, da, fa), (cb, db, fb) in zip(run(False), run(True)):
        assert (ca, da) == (cb, db)
        for x, y in zip(fa, fb):
            assert np.array_equal(x, y)


# one domain through the batch's X tiles of every shape and through the single-domain sweeps: FP32's
# arithmetic is the same in every kernel
@pytest.mark.gpu
@pytest.mark.parametrize("tile,cells_per_thread", [(128, 1), (256, 1), (512, 1), (256, 2), (512, 2)])
@pytest.mark.parametrize("test,nx,ny", [("Sod", 152, 98), ("Sod_circ", 256, 256)])
def test_fp32_batch_is_the_single_domain(armon, test, nx, ny, tile, cells_per_thread):
    kw = dict(max_cycles=6, precision=armon.PREC_FP32_MIXED, cfl=0.7, **GAD2)
    a, ca, da = _run(armon, test, nx=nx, ny=ny, **kw)
    spec = armon.ArmonDomainSpec(test=armon.TESTS[test], nx=nx, ny=ny, state=armon.reference_state(test))
    b = armon.Batch(armon.batch_params(verbose=5, **kw), [spec])
    b.set_tuning(16, tile_x=tile, x_cells_per_thread=cells_per_thread)
    b.init()
    b.begin()
    b.run()
    assert b.finish() == 0, armon.errors()
    assert (b.result(0).cycles, b.result(0).final_dt) == (ca, da)
    for f in FIELDS:
        assert np.array_equal(b.read(0, f), a[f]), f
    b.close()
