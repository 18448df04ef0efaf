"""Attempts that fail inside runs of steps, in every dimension and form of the
state, the 2D MHD ones (whose predictor parks its reference EMF in the next
faces' buffers) among them: each call has failures, and the halved retries
leave the oracle's states, faces, step and failure counts."""
import pytest

from helpers import gpu_grid, oracle_grid
from test_gpu_hydro3d import problem
from test_gpu_runs import PROBLEMS, same

pytestmark = pytest.mark.gpu

CASES = {"sod": 2.6, "kh": 3.5, "ot": 4.0, "turb": 3.5, "hydro3d": 4.0}


@pytest.mark.parametrize("name", sorted(CASES))
def test_failures_in_every_call(name):
    pb = list(problem((8, 7, 9)) if name == "hydro3d" else PROBLEMS[name]())
    pb[2] = dict(pb[2], cfl_coeff=CASES[name], verify_fallback=0)
    og, gg = oracle_grid(pb), gpu_grid(pb)
    failures = []
    for steps in (9, 4, 12):
        o = og.advance(1e9, True, steps)
        assert o == gg.advance(1e9, True, steps)
        failures.append(o[1])
        same(pb, og, gg)
    assert min(failures) > 0, failures
