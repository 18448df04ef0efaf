"""Steps launched ahead of the host (advance on grids without user
boundaries): the end of the time inside a run, more steps than one run holds,
failed attempts and their halved retries in the middle of one, a state without
signal speed, and the same grid advanced one call per step all match the
oracle's loop, step and failure counts included, bit for bit."""
import numpy as np
import pytest

import dragon_amd as D
from dragon_amd import problems as P

from helpers import compare_states, gpu_grid, oracle_grid

pytestmark = pytest.mark.gpu

PROBLEMS = {"sod": lambda: P.sod_1d(90), "kh": lambda: P.kelvin_helmholtz_2d(20), "ot": lambda: P.orszag_tang_2d(18),
            "turb": lambda: P.turbulence_3d(8)}


def pair(name, **switches):
    pb = PROBLEMS[name]()
    pb[2].update(switches)
    return pb, oracle_grid(pb), gpu_grid(pb)


def same(pb, og, gg):
    res = compare_states(gg, og, pb[0], 8 if pb[2]["mhd"] else 5)
    assert res["bit_equal"] and res.get("B_bit_equal", True), res


@pytest.mark.parametrize("name", sorted(PROBLEMS))
def test_frames_end_inside_runs(name):
    pb, og, gg = pair(name)
    og.advance(1e9, True, 1), gg.advance(1e9, True, 1)
    gg.apply_boundary()
    dt = gg.cfl_time()
    for frame in (0.3 * dt, 2.5 * dt, 11.2 * dt, 150.0 * dt if name in ("sod", "kh") else 3.0 * dt):
        assert og.advance(frame) == gg.advance(frame)
        same(pb, og, gg)


@pytest.mark.parametrize("name,coeff", [("sod", 2.6), ("kh", 3.5), ("ot", 2.5), ("turb", 2.5)])
def test_failed_attempts_inside_runs(name, coeff):
    """A CFL coefficient above the stable range: attempts fail and are halved."""
    pb, og, gg = pair(name, cfl_coeff=coeff, verify_fallback=0)
    total = 0
    for steps in (9, 4, 1, 12):
        o = og.advance(1e9, True, steps)
        g = gg.advance(1e9, True, steps)
        assert o == g
        total += o[1]
        same(pb, og, gg)
    print(name, "failed attempts", total)


@pytest.mark.parametrize("name", ["sod", "ot"])
def test_without_cfl_check(name):
    pb, og, gg = pair(name)
    og.advance(1e9, True, 1), gg.advance(1e9, True, 1)
    gg.apply_boundary()
    dt = 0.4 * gg.cfl_time()
    assert og.advance(dt, False) == gg.advance(dt, False) == (1, 0)
    same(pb, og, gg)


def test_no_signal_speed():
    pb = P.kelvin_helmholtz_2d(12)
    pb[4][..., 1:5] = 0.0
    gg = gpu_grid(pb)
    before = gg.get_w()
    with pytest.raises(D.DragonError) as e:
        gg.advance(1.0)
    assert e.value.code == D.DG_ERR_CFL and "max signal speed is zero" in str(e.value)
    g = gg.g
    assert np.array_equal(gg.get_w()[g:-g, g:-g], before[g:-g, g:-g])


def test_one_call_per_step_equals_one_run():
    pb = PROBLEMS["ot"]()
    a, b = gpu_grid(pb), gpu_grid(pb)
    for _ in range(70):
        a.advance(1e9, True, 1)
    assert b.advance(1e9, True, 70) == (70, 0)
    assert np.array_equal(a.get_w(), b.get_w()) and np.array_equal(a.get_B(), b.get_B())
