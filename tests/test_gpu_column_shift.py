"""The second-order advection along y over rows of whole blocks of 256 cells, above and below the sizes from
which it shifts its columns at the cost of a column of blocks: the whole range (more than the Infinity
Cache holds) and the same range cut in bands of rows that are too small for the shift, bit for bit, in
double and float."""
import ctypes as C

import numpy as np
import pytest

INPUTS = ("ustar", "rho", "umat", "vmat", "Emat")


@pytest.mark.gpu
@pytest.mark.parametrize("single", [False, True])
@pytest.mark.parametrize("nx,ny,ghosts", [(3072, 1230, 4), (3070, 1230, 5), (6400, 1200, 4), (2816, 1400, 4)])
def test_whole_and_in_bands(armon, single, nx, ny, ghosts):
    lib, host = (armon.load_f32() if single else armon.load()), armon.load()
    ny = 2 * ny if single else ny
    p = armon.make_params("Sod", scheme=1, projection=2, nx=nx, ny=ny, nb_ghosts=ghosts, engine=armon.ENGINE_STAGED,
                          verbose=5)
    host.armon_update_axis(C.byref(p), 1)
    rng = np.random.default_rng(nx)
    arrays = {f: armon.DeviceArray(p.nb_cells, f, rng.uniform(0.5, 2.0, p.nb_cells) - (f == "ustar"), single=single)
              for f in INPUTS}
    d = host.armon_domain_advection(C.byref(p))
    r, ir = armon.Range(), armon.InnerRange2D()
    host.armon_domain_iter2D(C.byref(d), C.byref(r), C.byref(ir))
    out = []
    for bands in (1, 7):
        to = [armon.DeviceArray(p.nb_cells, "out", np.zeros(p.nb_cells), single=single) for _ in range(4)]
        cuts = np.linspace(r.start, r.end, bands + 1).astype(np.int64)   # in the middle of rows
        for first, last in zip(cuts[:-1], cuts[1:]):
            part = armon.Range(int(first), int(last))
            lib.advection_second_order(C.byref(part), C.byref(ir), p.s, p.dx, 1e-4 / nx,
                                       *[C.byref(arrays[f].view) for f in INPUTS], *[C.byref(t.view) for t in to])
        out.append([t.download() for t in to])
        assert not armon.errors()
    for whole, banded in zip(*out):
        assert np.any(whole) and np.array_equal(whole, banded)
