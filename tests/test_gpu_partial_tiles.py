"""The interior's LDS tiles where they can go wrong, one RK4 step against the
oracle at every point: axes shorter than a tile, one point past whole tiles,
odd row and plane pitches (each parity has its own LDS layout; with an odd
point count every other field starts off 16-byte alignment), and boxes on
both sides of the tile-shape rule (8x8x4, 8x8x8 and 32x4x4, each pitch); per
patch and batched.  Tolerance 1e-12 of
each field's largest value: one step's rounding, as in the other step tests."""
import numpy as np
import pytest

from helpers import NF, random_state, rel_err

pytestmark = pytest.mark.gpu

SHAPES = [(7, 7, 7), (8, 7, 9), (9, 8, 7), (14, 14, 14), (15, 14, 15), (15, 15, 15), (16, 23, 11), (23, 17, 22),
          (22, 15, 31), (13, 40, 10), (70, 70, 71), (71, 71, 72), (78, 78, 71), (77, 77, 71)]


@pytest.mark.parametrize("shape,gauge", [(s, 0) for s in SHAPES] + [(s, 2) for s in SHAPES if max(s) < 60])
def test_one_step_on_partial_tiles_matches_oracle(orc, shape, gauge):
    import amssbssn as A
    h, dt = 0.5, 0.05
    p = A.PatchGeom(shape, (-1.0, -1.5, -2.0) + tuple(b + h * n for b, n in zip((-1.0, -1.5, -2.0), shape)), 3)
    X, Y, Z = p.coords()
    st = random_state(shape[::-1], seed=sum(shape), amp=0.01)
    U = [a.copy() for a in st]
    orc.step(U, X, Y, Z, p.bbox, dt, 0.02, 1e-5, gauge=gauge, bc=0, gw=3)
    for mode in (A.MODE_PLAIN, A.MODE_BATCHED):
        lv = A.Level([p], gauge=gauge, eps=0.02)
        lv.set_state(0, st)
        assert lv.step(dt, 1, mode, want_ham=A.RES_EVERY_STEP) == 0
        errs = [rel_err(lv.get_field(0, A.LIST_STATE, v), U[v]) for v in range(NF)]
        assert max(errs) <= 1e-12, (mode, errs)
        # a NaN in the last interior point is seen, whatever tile holds it
        bad = st[0].copy()
        bad[-4, -4, -4] = np.nan
        lv.set_field(0, A.LIST_STATE, 0, bad)
        assert lv.step(dt, 1, mode) == 1
        lv.close()
