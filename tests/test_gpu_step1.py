"""The 1D step in one pass (k_step1) against the oracle, bit for bit, at sizes
around its 62 cells a wavefront and 248 a workgroup; and the boundary list and
CFL tail of a run's step in one launch (k_bc_tail) against the loop that
launches them apart (live timing keeps it), ghosts included."""
import numpy as np
import pytest

import oracle as O

from test_gpu_boundary import cases, make_elements
from test_gpu_boundary_list import mixed

pytestmark = pytest.mark.gpu

STATE = O.s8(1.7, 0.9, 0.3, -0.2, 0.1, 0.5, -0.4, 0.25)


def random_state(wshape, mhd, seed):
    rng = np.random.default_rng(seed)
    w = 0.1 * rng.normal(0, 1, wshape)
    w[..., :2] = 1.0 + 0.5 * rng.random(wshape[:-1] + (2,))
    if not mhd:
        w[..., 5:] = 0.0
    return w


# cells with ghosts (2, or 3 with MHD): one less than, as many as and one more than 62 and 248, and the smallest
@pytest.mark.parametrize("mhd", [0, 1])
@pytest.mark.parametrize("total", [7, 61, 62, 63, 124, 247, 248, 249, 1000])
@pytest.mark.parametrize("limiter,muscl", [(0, 1), (2, 1), (1, 0)])
def test_1d_steps_match_oracle(total, mhd, limiter, muscl):
    import dragon_amd as D
    g = O.Grid((8,), (0.1,), O.Cfg(mhd=mhd, muscl=muscl, ctu=muscl), ghosts=1).g
    n = total - 2 * g
    cfg = dict(mhd=mhd, limiter=limiter, muscl=muscl, ctu=muscl)
    og = O.Grid((n,), (1.0 / n,), O.Cfg(**cfg), ghosts=1)
    gg = D.Grid((n,), (1.0 / n,), 1, D.Config(**cfg))
    w = random_state(og.wshape, mhd, total)
    og.set_w(w), gg.set_state(w, None)
    for steps in (1, 6):
        assert og.advance(1e9, True, steps) == gg.advance(1e9, True, steps)
        nf = 8 if mhd else 5
        assert np.array_equal(gg.get_w()[..., :nf], og.get_w()[..., :nf])


@pytest.mark.parametrize("mhd", [0, 1])
@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("shape", [(5,), (70,), (9, 67), (6, 5, 66)])
def test_boundary_and_tail_of_a_run(shape, precision, mhd):
    import dragon_amd as D
    dim = len(shape)
    for spec in cases(dim) + mixed(dim):
        out = []
        for apart in (False, True):
            gg = D.Grid(shape, (0.1,) * dim, 1, D.Config(mhd=mhd, precision=precision))
            w = random_state(gg.get_w().shape, mhd, sum(shape))
            B = 0.1 * np.random.default_rng(3).normal(0, 1, gg.get_B().shape) if gg.has_B else None
            gg.set_state(w, B)
            gg.boundary = D.BoundaryList(*make_elements(D, spec, STATE))
            if apart:
                gg.timing(1)
            counts = gg.advance(1e9, True, 4)
            out.append((counts, gg.t_advanced, gg.get_w(), gg.get_B() if B is not None else None))
        (c0, t0, w0, b0), (c1, t1, w1, b1) = out
        assert c0 == c1 and t0 == t1, (spec, c0, c1, t0, t1)
        nf = 8 if mhd else 5
        assert np.array_equal(w0[..., :nf], w1[..., :nf]), spec
        assert b0 is None or np.array_equal(b0, b1), spec
