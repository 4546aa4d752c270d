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
