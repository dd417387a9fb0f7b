"""The whole-array right-hand side (compute_rhs_dev) against the oracle, every
output at every point, where its tiles can go wrong: the smallest shapes, no
interior, partial tiles, odd row and plane pitches (with an odd point count
every other array starts off 16 bytes), symmetry planes, matter, and arrays
off 16 bytes on an even pitch.  Tolerance 1e-12 of each field's largest value,
as in the other right-hand-side tests."""
import numpy as np
import pytest

from helpers import grid, random_state, rel_err

pytestmark = pytest.mark.gpu

SHAPES = [(5, 5, 5), (6, 7, 5), (7, 8, 9), (14, 15, 13), (15, 15, 15), (15, 14, 17), (38, 21, 19), (37, 22, 18)]


def _device(st, off):
    import torch
    n = st[0].size
    buf = torch.zeros(len(st) * n + 1, dtype=torch.float64, device="cuda")
    t = buf[off:off + len(st) * n].view((len(st),) + st[0].shape)
    t.copy_(torch.tensor(np.stack(st)))
    return t


@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("co,gauge,off", [(0, 0, 0), (1, 2, 0), (0, 2, 1)])
@pytest.mark.parametrize("sym", [0, 2])
def test_rhs_matches_oracle(orc, shape, co, gauge, off, sym):
    from amssbssn import fortran_abi as fa
    nx, ny, nz = shape
    h = (0.3, 0.27, 0.33)
    X, Y, Z, _ = grid(nx, ny, nz, h, origin=(0.0, 0.0, 0.0) if sym else (-1.1, -0.9, -1.3))
    st = random_state((nz, ny, nx), seed=nx + ny + nz)
    rng = np.random.default_rng(5)
    mat = [0.05 * rng.standard_normal((nz, ny, nx)) for _ in range(10)]
    o = orc.compute_rhs(st, X, Y, Z, 0.02, co=co, symmetry=sym, gauge=gauge, matter=mat)
    d = (X[1] - X[0], Y[1] - Y[0], Z[1] - Z[0])
    g = fa.compute_rhs_dev(_device(st, off), d, 0.02, co=co, symmetry=sym, origin=(X[0], Y[0], Z[0]), gauge=gauge,
                           matter=_device(mat, off))
    assert g["flag"] == 0
    for key in ("rhs", "gam", "ric") + (("res",) if co == 0 else ()):
        for i, ref in enumerate(o[key]):
            e = rel_err(g[key][i].cpu().numpy(), ref)
            assert e <= 1e-12, (key, i, e)
    # a NaN in a corner, on a face and inside is reported
    for q in ((0, 0, 0), (nz - 1, ny // 2, 1), (nz // 2, ny // 2, nx // 2)):
        bad = [a.copy() for a in st]
        bad[3][q] = np.nan
        assert fa.compute_rhs_dev(_device(bad, off), d, 0.02, co=co, symmetry=sym, origin=(X[0], Y[0], Z[0]),
                                  gauge=gauge)["flag"] == 1
