"""A run's end, by the number of cycles and by time, for domains on both sides of the size from which a run
enqueues no more cycles than are left: the same cycles, time, time step and fields as the cycles advanced
one by one."""
import numpy as np
import pytest


@pytest.mark.gpu
@pytest.mark.parametrize("nx,ny", [(300, 40), (4096, 1024), (4100, 1025)])
@pytest.mark.parametrize("end", [dict(max_cycles=1), dict(max_cycles=16), dict(max_cycles=37), dict(max_time=2.5e-3)])
def test_run_ends_where_single_cycles_do(armon, nx, ny, end):
    kw = dict(nx=nx, ny=ny, scheme=1, projection=2, limiter=1, nb_ghosts=4, cfl=0.6, verbose=5,
              **{"max_cycles": 10**6, "max_time": 1e9, **end})
    r, s = armon.run(armon.make_params("Sod_circ", **kw))
    t = armon.Solver(armon.make_params("Sod_circ", graph_chunk=0, **kw))
    t.init_test()
    t.begin()
    t.advance(r.cycles + 3)
    q = t.finish()
    assert r.status == q.status == 0 and r.cycles >= 1
    assert (r.cycles, r.time, r.current_dt, r.final_dt) == (q.cycles, q.time, q.current_dt, q.final_dt)
    for f in ("rho", "umat", "vmat", "Emat", "pmat", "cmat"):
        assert np.array_equal(s.read(f), t.read(f)), f
    s.close()
    t.close()
