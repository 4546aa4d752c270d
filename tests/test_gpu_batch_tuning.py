"""A batch's launch configuration read and set again is the same configuration, Y tiles among it, and Y
tiles and marches can be chosen by hand for any batch, with the same bits."""
import numpy as np
import pytest

SCHEME = dict(scheme=1, projection=2, limiter=1, nb_ghosts=4, cfl=0.6, verbose=5, max_cycles=6)


def _key(t):
    return t.y_run_rows, t.grid_x, t.grid_y, t.items_x, t.items_y, t.y_tiles, t.tile_x, t.x_cells_per_thread


def _set(b, t, **kw):
    b.set_tuning(**{**dict(y_run_rows=t.y_run_rows, grid_x=t.grid_x, grid_y=t.grid_y, tile_x=t.tile_x,
                           x_cells_per_thread=t.x_cells_per_thread, y_tiles=bool(t.y_tiles)), **kw})


@pytest.mark.gpu
@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("autotune", [False, True])
def test_tuning_read_and_set_again(armon, precision, autotune):
    specs = armon.random_specs(31, 7, 24 * 24, 96 * 96)
    b = armon.Batch(armon.batch_params(precision=precision, **SCHEME), specs)
    b.init()
    t = b.autotune() if autotune else b.tuning()
    if not autotune:
        assert t.y_tiles and t.items_y == sum(-(-s.nx // 16) * -(-s.ny // 24) for s in specs)
    _set(b, t)
    assert _key(b.tuning()) == _key(t)
    c = armon.Batch(armon.batch_params(precision=precision, **SCHEME), specs)   # another batch
    _set(c, t)
    assert _key(c.tuning()) == _key(t)
    _set(c, c.tuning(), tile_x=128, x_cells_per_thread=1)   # one thing changed: the Y items stay
    assert (c.tuning().y_tiles, c.tuning().items_y) == (t.y_tiles, t.items_y)
    b.close()
    c.close()


@pytest.mark.gpu
@pytest.mark.parametrize("precision", [0, 1])
def test_tiles_by_hand_have_the_bits_of_marches(armon, precision):
    def run(y_tiles):
        b = armon.Batch(armon.batch_params(precision=precision, **SCHEME), armon.random_specs(8, 5, 20 * 20, 80 * 80))
        b.set_tuning(40, y_tiles=y_tiles)
        assert bool(b.tuning().y_tiles) == y_tiles
        b.init()
        b.begin()
        b.run()
        assert b.finish() == 0, armon.errors()
        out = [b.read(d, f) for d in range(b.n) for f in ("rho", "umat", "vmat", "Emat")]
        b.close()
        return out

    assert all(np.array_equal(x, y) for x, y in zip(run(True), run(False)))


@pytest.mark.gpu
@pytest.mark.parametrize("precision", [0, 1])
def test_autotune_leaves_the_initial_fields(armon, precision):
    """The fields between init and begin are init's, tuned or not; only the work arrays are the tuner's."""
    b = armon.Batch(armon.batch_params(precision=precision, **SCHEME), armon.random_specs(4, 3, 20 * 20, 60 * 60))
    b.init()
    fields = [f for f in armon.FIELD if not f.startswith("work")]
    before = [[b.read(d, f) for f in fields] for d in range(b.n)]
    b.autotune()
    for d in range(b.n):
        for f, x in zip(fields, before[d]):
            assert np.array_equal(b.read(d, f), x, equal_nan=True), (d, f)
    b.close()
