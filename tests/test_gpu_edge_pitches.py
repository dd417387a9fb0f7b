"""One RK4 step under the reference's boundary modes against the oracle, at
every point, on odd and even row and plane pitches (each parity has its own
window layout, and arrays with a symmetry plane their own kernel): shapes with
partial and single boundary tiles.  Tolerance 1e-12 of each field's largest
value, as in the other step tests."""
import pytest

from helpers import NF, random_state, rel_err

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", [(7, 7, 7), (8, 9, 7), (19, 17, 23), (23, 18, 20), (22, 19, 21), (39, 16, 11)])
@pytest.mark.parametrize("bc", [1, 2, 3])
@pytest.mark.parametrize("sym", [0, 1, 2])
def test_one_step_with_boundary_matches_oracle(orc, shape, bc, sym):
    import amssbssn as A
    h, dt = 0.5, 0.05
    lo = [0.0 if sym == 2 or (sym == 1 and a == 2) else -0.25 * h * n for a, n in enumerate(shape)]
    p = A.PatchGeom(shape, tuple(lo) + tuple(b + h * n for b, n in zip(lo, shape)), 3)
    X, Y, Z = p.coords()
    st = random_state(shape[::-1], seed=sum(shape) + bc, amp=0.01)
    gauge = 2 if bc == 1 else 0
    U = [a.copy() for a in st]
    orc.step(U, X, Y, Z, p.bbox, dt, 0.02, 1e-5, symmetry=sym, gauge=gauge, bc=bc, gw=3)
    for want in (A.RES_NONE, A.RES_EVERY_STEP):
        lv = A.Level([p], gauge=gauge, eps=0.02, bc=bc, symmetry=sym)
        lv.set_state(0, st)
        assert lv.step(dt, 1, want_ham=want) == 0
        errs = [rel_err(lv.get_field(0, A.LIST_STATE, v), U[v]) for v in range(NF)]
        lv.close()
        assert max(errs) <= 1e-12, (want, errs)
