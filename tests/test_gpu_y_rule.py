"""Flat and narrow domains on both sides of the rule that gives a Y sweep tiles or marches (y_takes_tiles in
armon-kokkos_amd/csrc/fused.hpp): the bits of marches of a given length, with the time step made in the
cycle's first sweep and by a kernel of its own, for one domain and in a batch."""
import numpy as np
import pytest

FIELDS = ("rho", "umat", "vmat", "Emat", "pmat", "cmat")
GAD2 = dict(scheme=1, projection=2, limiter=1, nb_ghosts=4)
GOD1 = dict(scheme=0, projection=1, nb_ghosts=2)


# Sequential starts along x, the symmetric splitting along y in its even cycles
@pytest.mark.gpu
@pytest.mark.parametrize("splitting", [0, 1, 2])
@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("nx,ny,scheme", [
    (75000, 4, GAD2), (40000, 8, GAD2), (9000, 25, GAD2), (16, 20000, GAD2), (5, 3001, GAD2), (100001, 3, GOD1),
    (30000, 29, GOD1), (3, 4099, GOD1)])
def test_flat_and_narrow_domains_have_the_bits_of_marches(armon, nx, ny, scheme, precision, splitting):
    def run(**more):
        r, s = armon.run(armon.make_params("Sod_circ", nx=nx, ny=ny, precision=precision, axis_splitting=splitting,
                                           max_cycles=5, cfl=0.5, verbose=5, **scheme, **more))
        assert r.status == 0, armon.errors()
        out = [s.read(f) for f in FIELDS]
        s.close()
        return out, r.cycles, r.final_dt

    (a, ca, da), (b, cb, db) = run(), run(y_run_rows=7)
    assert (ca, da) == (cb, db) and ca == 5
    for f, x, y in zip(FIELDS, a, b):
        assert np.array_equal(x, y), f


@pytest.mark.gpu
@pytest.mark.parametrize("sizes,tiles", [([(300000, 8)], 0), ([(60000, 4)] * 5, 0), ([(900, 800)], 1),
                                         ([(300, 200), (4000, 30), (30, 4000)], 1), ([(1620, 1620)], 0)])
def test_batch_starts_with_what_its_sizes_fill(armon, sizes, tiles):
    specs = [armon.ArmonDomainSpec(test=armon.TESTS["Sod"], nx=nx, ny=ny, state=armon.reference_state("Sod"))
             for nx, ny in sizes]

    def run(**tuning):
        b = armon.Batch(armon.batch_params(max_cycles=4, axis_splitting=1, cfl=0.5, verbose=5, **GAD2), specs)
        if tuning:
            b.set_tuning(**tuning)
        else:
            assert b.tuning().y_tiles == tiles
        b.init()
        b.begin()
        b.run()
        assert b.finish() == 0, armon.errors()
        out = [b.read(d, f) for d in range(b.n) for f in FIELDS]
        b.close()
        return out

    for x, y in zip(run(), run(y_run_rows=32, y_tiles=not tiles)):
        assert np.array_equal(x, y)


# narrow domains take tiles above the limit on cells too: 2.7 M and 3.9 M cells
@pytest.mark.gpu
@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("nx,ny,scheme", [(5, 780001, GAD2), (64, 61000, GOD1), (130, 30007, GAD2), (257, 15200, GOD1)])
def test_narrow_domains_above_the_limit(armon, nx, ny, scheme, precision):
    test_flat_and_narrow_domains_have_the_bits_of_marches(armon, nx, ny, scheme, precision, 1)


@pytest.mark.gpu
@pytest.mark.parametrize("nx,ny,tiles", [(5, 780001, 1), (40, 100000, 0), (64, 61000, 0), (1000, 3900, 0)])
def test_batch_of_a_narrow_domain(armon, nx, ny, tiles):
    spec = armon.ArmonDomainSpec(test=armon.TESTS["Sod"], nx=nx, ny=ny, state=armon.reference_state("Sod"))
    b = armon.Batch(armon.batch_params(max_cycles=4, verbose=5, **GAD2), [spec])
    assert b.tuning().y_tiles == tiles
    b.close()
