"""The smallest patches a batch takes (sides of 4 cells) against the oracle."""
import numpy as np
import pytest

from test_gpu_batch import build, oracle_patch

pytestmark = pytest.mark.gpu

SMALLEST = [(4, 4, 4.0, 0.2, 1.5), (4, 5, 3.0, 0.2, 1.2), (5, 4, 5.0, 0.25, 1.0), (4, 29, 4.0, 0.1, 1.5), (33, 4, 2.5, 0.1, 1.0),
            (5, 8, 3.5, 0.2, 1.4), (9, 33, 4.0, 0.1, 1.6)]


@pytest.mark.parametrize("graph", [False, True])
@pytest.mark.parametrize("bc", ["outflow", "periodic"])
def test_smallest_patches_match_oracle(bc, graph):
    """Sides of 4 cells with 3 ghosts, and sides around the tiles of 8 x 32
    points of the constrained-transport passes."""
    b, pbs = build(0, SMALLEST, bc=bc)
    for _ in range(2):
        b.run(3, graph=graph)
        b.sync()
    for p, pb in enumerate(pbs):
        G = oracle_patch(pb, bc)
        for _ in range(6):
            G.advance(1e9, True, 1)
        w, B = b.get_state(p)
        assert b.stats(p)["steps"] == 6
        assert np.array_equal(w, G.get_w()) and np.array_equal(B, G.get_B()), (pb[0], np.argwhere(w != G.get_w())[:5])
