"""The initial state of a batch, made by one launch over all its domains, against each domain's own
solver: every field, ghost cells included, bit for bit. Domains end anywhere in a wave of 64 cells and
start on the next one."""
import numpy as np
import pytest


@pytest.mark.gpu
@pytest.mark.parametrize("tests,sizes,ghosts", [
    (("Sod", "Sod_y", "Sod_circ", "Sedov"), [(4, 4), (57, 7), (64, 64), (100, 33), (5, 200)], 4),
    (("Bizarrium",), [(8, 8), (31, 17), (129, 3)], 5),
    (("Sedov",), [(24, 24)], 3)])
def test_initial_state(armon, tests, sizes, ghosts):
    kw = dict(scheme=0, projection=1, nb_ghosts=ghosts, max_cycles=2, verbose=5)
    specs, names = [], []
    for k, (nx, ny) in enumerate(sizes):
        name = tests[k % len(tests)]
        names.append(name)
        # Sedov's high region and energy go with the cell size
        option = armon.load().armon_test_option(armon.make_params(name, nx=nx, ny=ny, **kw))
        specs.append(armon.ArmonDomainSpec(test=armon.TESTS[name], nx=nx, ny=ny,
                                           state=armon.reference_state(name, option)))
    b = armon.Batch(armon.batch_params(**kw), specs)
    b.init()
    for d, (nx, ny) in enumerate(sizes):
        s = armon.Solver(armon.make_params(names[d], nx=nx, ny=ny, **kw))
        s.init_test()
        for f in armon.FIELD:
            if not f.startswith("work"):
                assert np.array_equal(b.read(d, f), s.read(f)), (names[d], nx, ny, f)
        s.close()
    b.close()
