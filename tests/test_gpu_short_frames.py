"""Frames of a single step (advance by less than the CFL step, as a caller
that couples the grid to something else does) take no longer than that step
with its boundary pass, its CFL step and the step itself called one by one;
half as long again is allowed for."""
import time

import numpy as np
import pytest

from dragon_amd import problems as P

from helpers import gpu_grid
from test_gpu_hydro3d import problem

pytestmark = pytest.mark.gpu

PROBLEMS = {"sod_1024": lambda: P.sod_1d(1024), "hydro3d_16": lambda: problem((16, 16, 16)), "hydro3d_64": lambda: problem((64, 64, 64)),
            "kh_700": lambda: P.kelvin_helmholtz_2d(700), "ot_128": lambda: P.orszag_tang_2d(128), "ot_1024": lambda: P.orszag_tang_2d(1024),
            "turb_96": lambda: P.turbulence_3d(96)}


@pytest.mark.parametrize("name", sorted(PROBLEMS))
def test_one_step_frame(name):
    gg = gpu_grid(PROBLEMS[name]())
    gg.advance(1e9, True, 2)
    gg.apply_boundary()
    dt = 0.3 * gg.cfl_time()

    def one_by_one():
        gg.apply_boundary()
        gg.unsplit_step(min(dt, gg.cfl_time()))

    def median(f):
        t = []
        for _ in range(15):
            t0 = time.perf_counter()
            f()
            t.append(time.perf_counter() - t0)
        return np.median(t[3:])

    apart, frame = median(one_by_one), median(lambda: gg.advance(dt))
    print(f"{name}: one by one {apart * 1e6:.0f} us, a frame {frame * 1e6:.0f} us")
    assert gg.advance(dt) == (1, 0)
    assert frame <= 1.5 * apart


@pytest.mark.parametrize("name", ["sod_1024", "ot_128", "turb_96"])
def test_one_step_without_cfl(name):
    """Without the CFL check one step takes all the time, whatever the limit
    on steps."""
    gg = gpu_grid(PROBLEMS[name]())
    gg.advance(1e9, True, 2)
    gg.apply_boundary()
    dt = 0.1 * gg.cfl_time()

    def median(f):
        t = []
        for _ in range(15):
            t0 = time.perf_counter()
            f()
            t.append(time.perf_counter() - t0)
        return np.median(t[3:])

    def one_by_one():
        gg.apply_boundary()
        gg.unsplit_step(dt)

    apart, frame = median(one_by_one), median(lambda: gg.advance(dt, False, 20))
    print(f"{name}: one by one {apart * 1e6:.0f} us, a frame {frame * 1e6:.0f} us")
    assert gg.advance(dt, False, 20) == (1, 0)
    assert frame <= 1.5 * apart
