"""kernel_times counts and times the kernels that ran: no time-step kernel where the cycle's first sweep makes
the time step (small domains without a run length of their own, splittings of two or three sweeps)."""
import pytest

SCHEME = dict(scheme=1, projection=2, limiter=1, nb_ghosts=4, cfl=0.5, verbose=5, max_cycles=100)


@pytest.mark.gpu
@pytest.mark.parametrize("kw,launches", [
    (dict(nx=200, ny=100), [6, 6, 0, 0]), (dict(nx=1200, ny=1200), [6, 6, 6, 0]),
    (dict(nx=200, ny=100, y_run_rows=16), [6, 6, 6, 0]), (dict(nx=200, ny=100, axis_splitting=3), [6, 0, 6, 0]),
    (dict(nx=200, ny=100, axis_splitting=2), [9, 9, 0, 0]), (dict(nx=90000, ny=4, axis_splitting=1), [6, 6, 3, 0])])
def test_solver_counts_its_launches(armon, kw, launches):
    s = armon.Solver(armon.make_params("Sod", **{**SCHEME, **kw}))
    s.init_test()
    s.begin()
    t = s.kernel_times(6)
    assert list(t.launches) == launches
    assert all((ms > 0) == (n > 0) for ms, n in zip(t.total_ms, t.launches))
    s.close()


@pytest.mark.gpu
@pytest.mark.parametrize("march,launches", [(False, [4, 4, 0, 0]), (True, [4, 4, 4, 0])])
def test_batch_counts_its_launches(armon, march, launches):
    b = armon.Batch(armon.batch_params(**SCHEME), armon.random_specs(3, 4, 40 * 40, 60 * 60))
    if march:
        b.set_tuning(16, grid_x=2)
    b.init()
    b.begin()
    t = b.kernel_times(4)
    assert list(t.launches) == launches
    assert all((ms > 0) == (n > 0) for ms, n in zip(t.total_ms, t.launches))
    b.close()
