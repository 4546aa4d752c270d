"""Where a run ends and what the calls after it answer, for runs that the host ends between chunks of
cycles without a cycle after the last."""
import numpy as np
import pytest

SCHEME = dict(scheme=1, projection=2, limiter=1, nb_ghosts=4, cfl=0.5, verbose=5)


# a constant time step may be negative: the end time is never reached, the count of cycles is (40 cycles are
# more than a chunk of 16)
@pytest.mark.gpu
@pytest.mark.parametrize("precision", [0, 1])
def test_negative_constant_time_step_runs_every_cycle(armon, po, oracle, precision):
    kw = dict(SCHEME, nx=64, ny=32, cst_dt=1, Dt=-1e-5, max_cycles=40, max_time=0.2)
    r, s = armon.run(armon.make_params("Sod_circ", precision=precision, **kw))
    assert r.status == 0 and r.cycles == 40, armon.errors()
    status, data, cycles, dt, _ = po.run(oracle, po.make_params(oracle, "Sod_circ", **kw))
    assert status == 0 and (cycles, dt) == (r.cycles, r.final_dt)
    mask = data.array("domain_mask") == 1
    for f in ("rho", "umat", "vmat", "Emat"):
        if precision == 0:
            assert np.array_equal(s.read(f)[mask], data.array(f)[mask]), f
        else:
            assert np.allclose(s.read(f)[mask], data.array(f)[mask], rtol=1e-4, atol=1e-5), f
    s.close()


@pytest.mark.gpu
def test_batch_with_a_negative_constant_time_step_runs_every_cycle(armon):
    b = armon.Batch(armon.batch_params(cst_dt=1, Dt=-1e-5, max_cycles=40, **SCHEME),
                    armon.random_specs(3, 3, 16 * 16, 32 * 32))
    b.init()
    b.begin()
    b.run()
    assert b.finish() == 0, armon.errors()
    assert [b.result(d).cycles for d in range(b.n)] == [40] * 3
    b.close()


# 16 and 32 cycles are whole chunks; 4.2 M cells enqueue no more cycles than are left
@pytest.mark.gpu
@pytest.mark.parametrize("cycles", [1, 16, 20, 32])
@pytest.mark.parametrize("areas", [(16 * 16, 32 * 32), (2060 * 2060, 2070 * 2070)])
def test_no_domain_is_active_after_a_run(armon, cycles, areas):
    b = armon.Batch(armon.batch_params(**dict(SCHEME, max_cycles=cycles)), armon.random_specs(3, 2, *areas))
    b.init()
    b.begin()
    b.advance(cycles + 1)
    b.finish()
    want = [b.result(d).cycles for d in range(2)]   # a small domain may reach its end time first
    assert max(want) == cycles
    for _ in range(2):
        b.init()
        b.begin()
        b.run()
        assert b.active() == 0
        b.advance(1)   # nothing left to do
        assert b.active() == 0
        assert b.finish() == 0, armon.errors()
        assert b.active() == 0
        assert [b.result(d).cycles for d in range(2)] == want
    b.init()
    b.begin()
    b.advance(1)
    assert b.active() == 2
    b.finish()
    b.close()
