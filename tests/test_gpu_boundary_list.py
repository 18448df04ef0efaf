"""Boundary lists that fit one launch (k_bc_list: at most one pass per face,
full transverse ranges, axes of ng + 2 cells or more) against the oracle's
pass-by-pass fill, bit for bit, on every list of the boundary tests and on
mixed lists: a different kind per face, in several orders, an axis left out."""
import itertools

import numpy as np
import pytest

import oracle as O

from test_gpu_boundary import FIX, GATED, IGN, OUT, PER, REF, X, XN, XP, Y, YN, YP, Z, ZN, ZP, add_oracle, cases, make_elements

pytestmark = pytest.mark.gpu

# the smallest axes the launch takes (5 with 3 ghosts), odd ones, one beyond a wavefront
SHAPES = {1: [(5,), (70,)], 2: [(5, 6), (9, 67)], 3: [(5, 6, 5), (6, 5, 66), (9, 80, 190)]}  # the last: a thread per ghost cell


def mixed(dim):
    out = []
    if dim >= 2:
        for p in itertools.permutations([(FIX, XN, True), (REF, YP, True), (PER, Z if dim == 3 else XP & 0, True), (OUT, XP | YN, True)]):
            out.append([e for e in p if e[1]])
        out += [[(REF, X, True), (GATED, Y, True)], [(GATED, Y, True), (REF, X, True)], [(PER, X, True), (FIX, Y, True)],
                [(FIX, Y, True), (PER, X, True)], [(FIX, XN, True), (FIX, YP, True)], [(IGN, X, True), (REF, Y, True)]]
    if dim == 3:
        out += [[(REF, ZN, True), (PER, Y, True), (FIX, ZP, True)], [(GATED, Z, True), (FIX, YN, True), (REF, X | YP, True)]]
    return out


@pytest.mark.parametrize("mhd", [0, 1])
@pytest.mark.parametrize("shape", [s for d in (1, 2, 3) for s in SHAPES[d]])
def test_lists_match_oracle(shape, mhd):
    import dragon_amd as D
    dim = len(shape)
    rng = np.random.default_rng(sum(shape) + mhd)
    state = O.s8(1.7, 0.9, 0.3, -0.2, 0.1, 0.5, -0.4, 0.25)
    for spec in cases(dim) + mixed(dim):
        og = O.Grid(shape, (0.1,) * dim, O.Cfg(mhd=mhd), ghosts=1)
        w = rng.normal(0, 1, og.wshape)
        w[..., :2] = np.abs(w[..., :2]) + 0.5
        if not mhd:
            w[..., 5:] = 0.0
        og.set_w(w)
        B = rng.normal(0, 1, og.bshape) if og.has_B else None
        if B is not None:
            og.set_B(B)
        add_oracle(og, spec, state)
        og.apply_bc()
        gg = D.Grid(shape, (0.1,) * dim, 1, D.Config(mhd=mhd))
        gg.set_state(w, B)
        gg.boundary = D.BoundaryList(*make_elements(D, spec, state))
        gg.apply_boundary()
        nf = 8 if mhd else 5
        wg, wo = gg.get_w()[..., :nf], og.get_w()[..., :nf]
        assert np.array_equal(wg, wo), (spec, np.argwhere(wg != wo)[:5])
        if B is not None:
            assert np.array_equal(gg.get_B(), og.get_B()), (spec, np.argwhere(gg.get_B() != og.get_B())[:5])
