"""dg_step_noalloc on 3D hydro, whose corner fluxes lie in another part of the
static scratch than the other grids' arrays: dg_step's next state, bit for
bit, in both precisions, a smaller grid after a larger one."""
import pytest

import dragon_amd as D

from test_gpu_hydro3d import problem
from test_zz_no_alloc import one_case


@pytest.mark.gpu
@pytest.mark.parametrize("precision", [D.FP64, D.MIXED])
@pytest.mark.parametrize("ctu", [0, 1])
def test_noalloc_matches_step(ctu, precision):
    import torch
    for shape in ((21, 18, 26), (5, 7, 6)):
        one_case(problem(shape, ctu=ctu), precision, torch)
