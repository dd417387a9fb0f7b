"""The 32x4x4 interior tiles where they can go wrong, one RK4 step and its
seven constraint norms against the oracle.  In the batched step's lists (tile
shape 3, one workgroup per tile and persistent): a last tile of 27 to 31 points
along x, rows that end in 8x8x8 tiles, y and z that are no multiple of 4.  In
the single-patch step: odd row pitches and both gauges, on a box that both
covers pad alike.  Tolerance 1e-12 of each field's largest value and 1e-12 of
each norm, as in the other step and norm tests."""
import numpy as np
import pytest

from helpers import NF, random_state, rel_err

pytestmark = pytest.mark.gpu


def _step(orc, shape, gauge):
    import amssbssn as A
    h = 0.5
    lo = (-1.0, -1.5, -2.0)
    p = A.PatchGeom(shape, lo + tuple(b + h * n for b, n in zip(lo, shape)), 3)
    X, Y, Z = p.coords()
    st = random_state(shape[::-1], seed=11 * sum(shape), amp=0.01)
    U = [a.copy() for a in st]
    orc.enforce_ga(U)
    res = orc.compute_rhs(U, X, Y, Z, 0.02, co=0, gauge=gauge)["res"]
    s = np.s_[3:-3, 3:-3, 3:-3]
    norms = np.array([np.sqrt(np.sum(r[s] ** 2) * h ** 3) for r in res])
    U = [a.copy() for a in st]
    orc.step(U, X, Y, Z, p.bbox, 0.05, 0.02, 1e-5, gauge=gauge, bc=0, gw=3)
    return p, st, U, norms


def _check(p, st, U, norms, gauge, mode, tune=None):
    import amssbssn as A
    lv = A.Level([p], gauge=gauge, eps=0.02)
    lv.set_state(0, st)
    if tune is not None:
        lv.set_tune(*tune)
    assert lv.step(0.05, 1, mode, want_ham=A.RES_EVERY_STEP) == 0
    errs = [rel_err(lv.get_field(0, A.LIST_STATE, v), U[v]) for v in range(NF)]
    got = lv.constraint_series()[0]
    lv.close()
    assert max(errs) <= 1e-12, (tune, errs)
    assert np.max(np.abs(got / norms - 1.0)) <= 1e-12, (tune, got, norms)


@pytest.mark.parametrize("shape", [(34, 15, 17), (36, 16, 11), (66, 15, 16), (44, 13, 15)])
@pytest.mark.parametrize("gauge", [0, 2])
def test_partial_wide_tiles_of_a_list_match_oracle(orc, shape, gauge):
    import amssbssn as A
    c = _step(orc, shape, gauge)
    for tune in ((3, 0, 1), (3, 0, 0), (3, 24, 1)):
        _check(*c, gauge, A.MODE_BATCHED, tune)


@pytest.mark.parametrize("shape", [(101, 69, 51), (102, 69, 51)])
@pytest.mark.parametrize("gauge", [0, 2])
def test_wide_tiles_of_a_patch_match_oracle(orc, shape, gauge):
    import amssbssn as A
    _check(*_step(orc, shape, gauge), gauge, A.MODE_PLAIN)
