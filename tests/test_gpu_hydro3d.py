"""3D hydro: the sweeps that rebuild the half states (corner fluxes two at a
time) and the reference-structured path (DG_UNFUSED) against the oracle, bit
for bit, CTU on and off, at sizes around the walkers' and wavefronts' ends;
the mixed form, which solves the predictor and corner fluxes in FP64, within
the bar of the mixed form."""
import numpy as np
import pytest

import dragon_amd as D
from dragon_amd import problems as P

from helpers import compare_states, gpu_grid, interior, oracle_grid, rel_l1

pytestmark = pytest.mark.gpu


def problem(shape, limiter=2, ctu=1, bcs=((1, 63),)):
    pb = P.diagonal_3d(4, limiter)
    g, rng = 2, np.random.default_rng(sum(shape))
    w = np.zeros(tuple(s + 2 * g for s in shape) + (8,))
    wi = interior(w, g, shape)
    wi[..., 0] = 1 + 0.5 * rng.random(shape)
    wi[..., 1] = 1 + 0.5 * rng.random(shape)
    wi[..., 2:5] = rng.normal(0, 0.5, shape + (3,))
    return shape, tuple(1 / s for s in shape), dict(pb[2], ctu=ctu, limiter=limiter), list(bcs), w, None, {}


@pytest.mark.parametrize("ctu", [0, 1])
@pytest.mark.parametrize("shape", [(1, 2, 3), (4, 5, 61), (5, 4, 62), (9, 33, 64), (34, 7, 66)])
@pytest.mark.parametrize("unfused", [False, True])
def test_matches_oracle(shape, ctu, unfused, monkeypatch):
    if unfused:
        monkeypatch.setenv("DG_UNFUSED", "1")
    pb = problem(shape, ctu=ctu, bcs=((0, 63),) if min(shape) < 3 else ((1, 63),))
    og, gg = oracle_grid(pb), gpu_grid(pb)
    assert og.advance(1e9, True, 4) == gg.advance(1e9, True, 4)
    assert compare_states(gg, og, shape, 5)["bit_equal"]


@pytest.mark.parametrize("chunk", [1, 5])
def test_walker_lengths(chunk, monkeypatch):
    pb = problem((23, 18, 40))
    og = oracle_grid(pb)
    monkeypatch.setenv("DG_MARCH_CHUNK", str(chunk))
    gg = gpu_grid(pb)
    assert og.advance(1e9, True, 3) == gg.advance(1e9, True, 3)
    assert compare_states(gg, og, pb[0], 5)["bit_equal"]


@pytest.mark.parametrize("ctu", [0, 1])
def test_mixed(ctu):
    pb = problem((30, 22, 41), ctu=ctu)
    og, gg = oracle_grid(pb), gpu_grid(pb, D.MIXED)
    og.advance(1e9, True, 4), gg.advance(1e9, True, 4)
    a, b = interior(gg.get_w(), 2, pb[0])[..., :5], interior(og.get_w(), 2, pb[0])[..., :5]
    assert np.all(rel_l1(a, b) < 1e-5)
