"""Modes of Psi4 on spheres of few points, whose last (or only) workgroup of
the interpolation is partly filled: 8, 32, 72 and 1,568 points without
symmetry, halves and eighths of that with it, against the oracle.  The same
tableaux in the same order, then sums of at most 1,568 points: relative to
the largest mode, 1e-12, as for the larger spheres."""
import numpy as np
import pytest

from test_oracle_surface import SOA_I, SOA_R, _fields, _grid, _mesh

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("sym", [0, 1, 2])
@pytest.mark.parametrize("nquarter", [1, 2, 3, 14])
def test_small_spheres_match_oracle(orc, sym, nquarter):
    import torch
    import amssbssn.fortran_abi as F
    X, Y, Z = _grid(sym)
    fields = _fields(*_mesh(X, Y, Z), sym)
    dev = [torch.tensor(np.ascontiguousarray(a), dtype=torch.float64, device="cuda:0") for a in fields]
    rp, ip = F.surf_wave_dev(*dev, X, Y, Z, 2.5, nquarter, 4, soa_r=SOA_R, soa_i=SOA_I, symmetry=sym)
    rc, orp, oip = orc.surf_wave(*fields, X, Y, Z, 2.5, nquarter, 4, soa_r=SOA_R, soa_i=SOA_I, symmetry=sym)
    assert rc == 0
    want = orp + 1j * oip
    assert np.max(np.abs(rp + 1j * ip - want)) <= 1e-12 * np.max(np.abs(want))
