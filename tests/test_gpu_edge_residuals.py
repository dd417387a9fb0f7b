"""The constraint residuals of a predictor at every point against the oracle,
under the boundary modes that use the boundary stencils: odd and even row and
plane pitches, with and without symmetry planes (the mirror image of a tile's
window is written in LDS), boundary tiles at the planes' corners included.
The oracle's residuals are those of its right-hand side (co = 0) on the step's
enforced base state.  Tolerance 1e-12 of each residual's largest value, as for
the right-hand side itself: enforce_ga's rounding, some 1e-16 of metric values
near 1, enters second differences of weight 5 / h^2 = 21 and residuals of
about 0.1, which leaves a factor of 50."""
import pytest

from helpers import random_state, rel_err

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", [(7, 7, 7), (15, 14, 13), (14, 15, 13), (15, 15, 15), (23, 18, 20), (39, 16, 11)])
@pytest.mark.parametrize("bc,gauge", [(2, 0), (3, 2)])
@pytest.mark.parametrize("sym", [0, 1, 2])
def test_predictor_residuals_match_oracle_at_every_point(orc, shape, bc, gauge, sym):
    import amssbssn as A
    h = 0.5
    lo = [0.0 if sym == 2 or (sym == 1 and a == 2) else -0.25 * h * n for a, n in enumerate(shape)]
    p = A.PatchGeom(shape, tuple(lo) + tuple(b + h * n for b, n in zip(lo, shape)), 3)
    X, Y, Z = p.coords()
    st = random_state(shape[::-1], seed=7 * sum(shape) + bc, amp=0.01)
    U = [a.copy() for a in st]
    orc.enforce_ga(U)
    want = orc.compute_rhs(U, X, Y, Z, 0.02, co=0, symmetry=sym, gauge=gauge)["res"]
    lv = A.Level([p], gauge=gauge, eps=0.02, bc=bc, symmetry=sym)
    lv.set_state(0, st)
    assert lv.step(0.05, 1, want_ham=A.RES_EVERY_STEP) == 0
    errs = [rel_err(lv.get_field(0, A.LIST_RES, a), want[a]) for a in range(7)]
    lv.close()
    assert max(errs) <= 1e-12, errs
