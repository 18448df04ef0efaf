"""The kernels' own FP64 quotients and square roots (Den, dsqrt in
dg_math.hpp) round like the CPU's over the range they are used in: states
whose density and pressure are scaled far up and down (B with the square
root, velocities kept) step bit for bit like the oracle."""
import math

import pytest

from dragon_amd import problems as P

from helpers import compare_states, gpu_grid, oracle_grid

pytestmark = pytest.mark.gpu

PROBLEMS = {"mhd_hlld": lambda: P.rotor_2d(21, 4.0, 0.12, 1.5, ny=18), "hydro_hllc": lambda: P.kelvin_helmholtz_2d(24),
            "mhd_3d": lambda: P.turbulence_3d(10), "hydro_1d": lambda: P.sod_1d(70)}


@pytest.mark.parametrize("scale", [1e-60, 1e-7, 1e60])
@pytest.mark.parametrize("name", sorted(PROBLEMS))
def test_scaled_states_bit_exact(name, scale):
    pb = PROBLEMS[name]()
    shape, d, cfg, bcs, w, B, meta = pb
    w[..., 0:2] *= scale
    w[..., 5:8] *= math.sqrt(scale)
    if B is not None:
        B *= math.sqrt(scale)
    og, gg = oracle_grid(pb), gpu_grid(pb)
    assert og.advance(1e9, True, 3) == gg.advance(1e9, True, 3)
    res = compare_states(gg, og, shape, 8 if cfg["mhd"] else 5)
    assert res["bit_equal"] and res.get("B_bit_equal", True), res
