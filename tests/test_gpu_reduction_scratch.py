"""A CFL bound that is still on its way on one stream while the conservation sums run on another: both as
they are alone."""
import ctypes as C

import numpy as np
import pytest


@pytest.mark.gpu
@pytest.mark.parametrize("nx,ny", [(61, 37), (1500, 1100)])
def test_cfl_bound_and_conservation_sums_on_two_streams(armon, nx, ny):
    lib = armon.load()
    solvers = [armon.Solver(armon.make_params("Sod", nx=16, ny=16, verbose=5)) for _ in range(2)]   # their streams
    streams = [lib.armon_solver_stream(s.h) for s in solvers]
    p = armon.make_params("Sod", nx=nx, ny=ny, engine=armon.ENGINE_STAGED, verbose=5)
    rng = np.random.default_rng(7)
    a = {f: armon.DeviceArray(p.nb_cells, f, rng.uniform(0.5, 2.0, p.nb_cells))
         for f in ("rho", "umat", "vmat", "Emat", "cmat", "domain_mask")}
    d = lib.armon_real_domain(C.byref(p))
    r, ir = armon.Range(), armon.InnerRange1D()
    lib.armon_domain_iter1D(C.byref(d), C.byref(r), C.byref(ir))
    view = lambda f: C.byref(a[f].view)  # noqa: E731
    calls = 60
    out = [armon.DeviceArray(1) for _ in range(calls)]

    def sums():
        mass, energy = C.c_double(), C.c_double()
        lib.conservation_vars(C.byref(r), C.byref(ir), 0.5, view("rho"), view("Emat"), view("domain_mask"),
                              C.byref(mass), C.byref(energy))
        return mass.value, energy.value

    def bound(at):
        lib.dt_CFL_device(C.byref(r), C.byref(ir), 0.5, 0.25, view("umat"), view("vmat"), view("cmat"),
                          view("domain_mask"), at.ptr)

    before = lib.armon_get_stream()
    try:
        want = sums()
        bound(out[0])
        lib.armon_synchronize()
        dt = out[0].download()[0]
        assert 0 < dt < 1
        for k in range(calls):
            lib.armon_set_stream(streams[0])
            bound(out[k])
            lib.armon_set_stream(streams[1])
            assert sums() == want, k
        lib.armon_set_stream(streams[0])
        lib.armon_synchronize()
    finally:
        lib.armon_set_stream(before)
    assert not armon.errors()
    assert [o.download()[0] for o in out] == [dt] * calls
    for s in solvers:
        s.close()
