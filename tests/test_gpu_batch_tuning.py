"""The tuner on a batch whose untuned tile is the best one keeps it."""
import pytest

from test_gpu_batch import build

pytestmark = pytest.mark.gpu


def test_tuning_keeps_the_untuned_tile_where_it_is_best():
    """One patch of 60 x 60: a face per thread, the untuned tile, takes 89 us
    a step, the next best tile 102."""
    b, _ = build(0, [(60, 60, 4.0, 0.1, 1.5)])
    assert b.tiles()[0] == 1
    tiles, _ = b.autotune(reps=40)
    assert tiles[0] == 1
