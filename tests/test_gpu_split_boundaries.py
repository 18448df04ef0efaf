"""Split steps with boundary lists whose second application changes what the
first one left (axes shorter than their ghosts, elements without corner
ghosts, two elements on a face): advance applies the list before its CFL step
and again before each sweep, as the oracle does, so every cell, ghosts
included, is the oracle's bit for bit."""
import numpy as np
import pytest

import dragon_amd as D
import oracle as O

from helpers import KIND, oracle_cfg
from test_gpu_split_sizes import problem

pytestmark = pytest.mark.gpu

ALL = {2: 15, 3: 63}
LISTS = {"reflective": lambda f: [(2, f, True)], "reflective, no corners": lambda f: [(2, f, False)],
         "periodic, no corners": lambda f: [(1, f, False)], "corners on x only": lambda f: [(2, 3, True), (1, f & 12, False)],
         "y first": lambda f: [(1, f & 12, False), (2, 3, False)], "two on a face": lambda f: [(2, 1, True), (0, 3, True), (1, 12, True)]}
CLS = {0: D.Outflow, 1: D.Periodic, 2: D.Reflective}


@pytest.mark.parametrize("shape", [(1, 20), (20, 1), (1, 1), (2, 2), (12, 10), (1, 5, 6), (5, 1, 4), (5, 6, 7)])
@pytest.mark.parametrize("name", sorted(LISTS))
def test_matches_oracle(name, shape):
    shape, d, cfg, _, w, _, _ = problem(shape, [])
    og = O.Grid(shape, d, oracle_cfg(cfg), ghosts=1)
    og.set_w(w)
    conf = D.Config()
    for k, v in cfg.items():
        setattr(conf, k, v)
    gg = D.Grid(shape, d, 1, conf)
    gg.set_state(w, None)
    els = []
    for kind, faces, corners in LISTS[name](ALL[len(shape)]):
        og.add_bc(KIND[kind], faces, corners, False, None)
        els.append(CLS[kind](faces, corners))
    gg.boundary = D.BoundaryList(*els)
    for steps in (1, 2, 5):
        assert og.advance_split(1e9, True, steps) == gg.advance_split(1e9, True, steps)
        a, b = gg.get_w()[..., :5], og.get_w()[..., :5]
        assert np.array_equal(a, b), (steps, np.argwhere(a != b)[:5])
