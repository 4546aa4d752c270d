"""boundary_conditions with its layers dealt to lanes (displacements of 1 and -1) or blocks, against the
layers filled one after the other on the host, bit for bit, in double and float: tall and flat domains,
numbers of layers around the lanes' 16, ranges that start late, and a displacement of 0."""
import ctypes as C

import numpy as np
import pytest

FIELDS = ("rho", "umat", "vmat", "pmat", "cmat", "gmat", "Emat")


@pytest.mark.gpu
@pytest.mark.parametrize("single", [False, True])
@pytest.mark.parametrize("nx,ny,ghosts,layers,start,stop", [
    (7, 30000, 4, 4, 0, None), (30000, 7, 4, 3, 0, None), (40, 33, 20, 1, 0, None), (40, 33, 20, 5, 2, 30),
    (40, 300, 20, 16, 0, None), (40, 300, 20, 17, 7, 299), (45, 45, 20, 20, 0, None), (64, 64, 4, 2, 63, None),
    (9, 70001, 2, 2, 5, None)])
def test_layers(armon, single, nx, ny, ghosts, layers, start, stop):
    lib = armon.load_f32() if single else armon.load()
    dtype = np.float32 if single else np.float64
    p = armon.make_params("Sod", nx=nx, ny=ny, nb_ghosts=ghosts, engine=armon.ENGINE_STAGED, verbose=5)
    rng = np.random.default_rng(nx + ny)
    for side in (0, 1, 2, 3):
        host = {f: rng.uniform(0.5, 2.0, p.nb_cells).astype(dtype) for f in FIELDS}
        dev = {f: armon.DeviceArray(p.nb_cells, f, host[f], single=single) for f in FIELDS}
        disp = C.c_int()
        d = armon.load().armon_boundary_conditions_domain(C.byref(p), side, C.byref(disp))
        r, ir = armon.Range(), armon.InnerRange1D()
        armon.load().armon_domain_direct_iter1D(C.byref(d), C.byref(r), C.byref(ir))
        r.start, r.end = min(start, r.end - 1), r.end if stop is None else min(stop, r.end)   # within the border
        for shift in (disp.value, 0):
            if shift == 0 and layers > 5:
                continue
            lib.boundary_conditions(C.byref(r), C.byref(ir), layers, shift, -0.75, 0.5,
                                    *[C.byref(dev[f].view) for f in FIELDS])
            at = np.arange(r.start, r.end) * ir.step + ir.start
            for w in range(layers):
                to, of = at - w * shift, at + (w + 1) * shift
                for f in FIELDS:
                    factor = dtype({"umat": -0.75, "vmat": 0.5}.get(f, 1.0))
                    host[f][to] = host[f][of] * factor
            lib.armon_synchronize()
            assert not armon.errors()
            for f in FIELDS:
                assert np.array_equal(dev[f].download(), host[f]), (side, shift, f)
