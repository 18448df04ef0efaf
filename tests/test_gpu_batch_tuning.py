"""The tuner keeps the untuned tile of a batch where it is the best one; the
mixed form's results do not depend on the tiles."""
import numpy as np
import pytest

from test_gpu_batch import build

pytestmark = pytest.mark.gpu


def test_tuning_keeps_the_untuned_tile_where_it_is_best():
    """One patch of 60 x 60: a face per thread, the untuned tile, takes 89 us
    a step, the next best tile 102."""
    b, _ = build(0, [(60, 60, 4.0, 0.1, 1.5)])
    assert b.tiles()[0] == 1
    b.run(200)  # the clock is up before anything is timed
    b.sync()
    tiles, _ = b.autotune(reps=40)
    assert tiles[0] == 1


def test_mixed_results_do_not_depend_on_the_shapes():
    ref = None
    for tile, width in ((1, 64), (5, 32), (32, 16), (4, 0)):
        b, pbs = build(1)
        b.set_tiles([tile] * 4)
        b.set_ysweep([width] * 4)
        b.run(6)
        b.sync()
        got = [b.get_state(p) for p in range(len(pbs))]
        ref = ref or got
        for p, ((w, B), (w0, B0)) in enumerate(zip(got, ref)):
            assert np.array_equal(w, w0) and np.array_equal(B, B0), (tile, width, p)
