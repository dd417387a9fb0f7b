"""prolong3 / restrict3 against the oracle at the edges of their tiles (32 x 8
x 8 fine, 16 x 4 x 4 coarse cells): extents one below, at and one past whole
tiles, target regions starting on odd and even fine cells, mirrored halo
reads.  Tolerance 1e-14 of the array's largest value: the same summation
order, contracted with FMAs."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nf", [(31, 7, 9), (32, 8, 8), (33, 9, 17), (65, 16, 15), (64, 33, 24)])
@pytest.mark.parametrize("off", [0, 1, 2, 5])
@pytest.mark.parametrize("start", [0, 1])
def test_transfer_tile_edges_match_oracle(orc, nf, off, start):
    from amssbssn import fortran_abi as fa
    rng = np.random.default_rng(sum(nf) + off)
    CD, FD = 0.5, 0.25
    nc = [(n + off) // 2 + 5 for n in nf]
    llbc = np.array([0.25, -1.0, 0.0])
    llbf = llbc + FD * off                       # off 0 and 1 read the mirrored halo
    uubc, uubf = llbc + CD * np.array(nc), llbf + FD * np.array(nf)
    func, funf = rng.standard_normal(nc[::-1]), rng.standard_normal(nf[::-1])
    soa = (1.0, -1.0, 1.0)
    lo, hi = llbf + FD * start, uubf
    o, g = funf.copy(), funf.copy()
    rc = orc.prolong3(func, llbc, uubc, o, llbf, uubf, lo, hi, soa)
    assert fa.prolong3(func, llbc, uubc, g, llbf, uubf, lo, hi, soa) == rc == 0
    assert np.max(np.abs(g - o)) <= 1e-14 * np.max(np.abs(o)) and np.array_equal(g == funf, o == funf)
    # the coarse cells whose stencils lie in the fine array and its halo
    c0, c1 = [(off + 1) // 2 + 1 + start] * 3, [(n + off) // 2 - 2 for n in nf]
    if min(b - a for a, b in zip(c0, c1)) < 1:
        return
    lo, hi = llbc + CD * np.array(c0), llbc + CD * np.array(c1)
    o, g = func.copy(), func.copy()
    if orc.restrict3(o, llbc, uubc, funf, llbf, uubf, lo, hi, soa):
        return
    fa.restrict3(g, llbc, uubc, funf, llbf, uubf, lo, hi, soa)
    assert np.max(np.abs(g - o)) <= 1e-14 * np.max(np.abs(o)) and np.array_equal(g == func, o == func)
    assert not np.array_equal(g, func)
