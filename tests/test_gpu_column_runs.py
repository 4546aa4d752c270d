"""The fluxes and the second-order advection along y shift the columns of a run so that its waves start on
lines, or do not, by the length of the row: at the edges of that rule (rows around whole blocks of 256
cells, 11 to 25 of them; ghost layers that put a row's start anywhere in a line), over whole and cut
ranges, bit for bit against the oracle."""
import ctypes as C

import pytest

from test_gpu_stages import ADV, SEED, Case, domain, it2d

pytestmark = pytest.mark.gpu
GAD = ["ustar", "pstar", "rho", "u", "pmat", "cmat"]


@pytest.mark.parametrize("nx,ny,g", [(237, 21, 4), (241, 20, 5), (242, 9, 4), (256, 17, 4), (257, 17, 7),
                                     (2816, 9, 4), (3072, 10, 5), (6144, 9, 4), (6400, 9, 5)])
@pytest.mark.parametrize("cut", ["full", "partial"])
def test_runs_of_shifted_columns(armon, po, oracle, nx, ny, g, cut):
    lib = armon.load()
    p = domain(armon, axis=1, nx=nx, ny=ny, g=g)
    for names, entry, want, region, last in (
            (GAD, lib.acoustic_GAD, oracle.o_acoustic_GAD, lib.armon_domain_fluxes, (1,)),
            (ADV, lib.advection_second_order, oracle.o_advection_second_order, lib.armon_domain_advection, ())):
        c = Case(armon, p.nb_cells, names, seed=SEED + nx + g)
        r, ir, orr, oir = it2d(armon, po, region(C.byref(p)))
        if cut == "partial":
            n = ir.row_range_length
            r.start, r.end = n // 3 + n, r.end - n // 2
            orr.start, orr.end = r.start, r.end
        args = (0.0071, p.dx) if names is GAD else (p.dx, 0.0071)
        entry(C.byref(r), C.byref(ir), p.s, *args, *[c.v(k) for k in names], *last)
        want(C.byref(orr), C.byref(oir), p.s, *args, *[c.h(k) for k in names], *last)
        c.compare(names[:2] if names is GAD else names[5:])
