"""Grids large enough for a launch per sweep axis (smaller ones sweep all axes
in one launch): one step of each physics against the oracle, bit for bit."""
import numpy as np
import pytest

from dragon_amd import problems as P

from helpers import compare_states, gpu_grid, oracle_grid

pytestmark = pytest.mark.gpu


def turbulent(shape, mhd):
    rng = np.random.default_rng(5)
    g = 3 if mhd else 2
    w = np.zeros(tuple(s + 2 * g for s in shape) + (8,))
    wi = w[tuple(slice(g, g + s) for s in shape)]
    wi[..., 0] = 1 + 0.3 * rng.random(shape)
    wi[..., 1] = 1 + 0.3 * rng.random(shape)
    for q in range(len(shape)):  # smooth along one axis, rough along the others
        wi[..., 2 + q] = 0.5 * rng.standard_normal(shape[0]).reshape((-1,) + (1,) * (len(shape) - 1))
    B = None
    if mhd:
        B = np.zeros(tuple(s + 1 + 2 * g for s in shape) + (3,))
        B[..., 0] = 0.4
        B[..., 1] = 0.3
    cfg = dict(mhd=int(mhd), gamma=5 / 3, solver=5, limiter=2, ctu=1, ct_energy=2)
    return shape, tuple(1 / s for s in shape), cfg, [(1, 63)], w, B, {"init_B": mhd}


@pytest.mark.parametrize("shape,mhd", [((2101, 2090), False), ((2101, 2090), True), ((161, 160, 150), False), ((161, 160, 150), True)])
def test_one_step(shape, mhd):
    pb = turbulent(shape, mhd)
    og, gg = oracle_grid(pb, 16), gpu_grid(pb)
    print("start", shape, mhd, flush=True)
    assert og.advance(1e9, True, 1) == gg.advance(1e9, True, 1)
    res = compare_states(gg, og, shape, 8 if mhd else 5)
    assert res["bit_equal"] and res.get("B_bit_equal", True), res
