"""amss_level_copy_list against the level's own grid functions, bit for bit:
even and odd point counts (16- and 8-byte copies), arrays off 16-byte
alignment, and the calls that must keep the effect of 24 copies in order
(outputs that share an array, arrays of the level itself)."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _copy(A, lv, lst, ptrs, d):
    return A.lib().amss_level_copy_list(lv.h, 0, lst, (C.c_void_p * 24)(*ptrs), d)


@pytest.mark.parametrize("shape", [(7, 7, 7), (8, 7, 9), (22, 22, 22), (41, 33, 27)])
@pytest.mark.parametrize("off", [0, 1])
def test_copy_list_in_and_out(shape, off):
    import torch
    import amssbssn as A
    lv = A.Level([A.PatchGeom(shape, (0.0, 0.0, 0.0) + tuple(0.5 * n for n in shape))])
    n = int(np.prod(shape))
    s = torch.cuda.ExternalStream(lv.stream())
    src = torch.randn(24 * n + 1, dtype=torch.float64, device="cuda")[off:off + 24 * n]
    dst = torch.zeros(24 * n + 1, dtype=torch.float64, device="cuda")[off:off + 24 * n]
    torch.cuda.synchronize()
    ptr = lambda t: [t.data_ptr() + 8 * n * v for v in range(24)]  # noqa: E731
    assert _copy(A, lv, A.LIST_STATE, ptr(src), 0) == 0
    assert _copy(A, lv, A.LIST_STATE, ptr(dst), 1) == 0
    s.synchronize()
    assert torch.equal(src, dst)
    got = np.stack([lv.get_field(0, A.LIST_STATE, v).ravel() for v in range(24)])
    assert np.array_equal(got, src.cpu().numpy().reshape(24, n))
    # outputs that share one array: the last field's values stay
    one = torch.zeros(n, dtype=torch.float64, device="cuda")
    torch.cuda.synchronize()
    assert _copy(A, lv, A.LIST_STATE, [one.data_ptr()] * 24, 1) == 0
    s.synchronize()
    assert np.array_equal(one.cpu().numpy(), got[23])
    # arrays of the level: another list, and the list itself shifted by one field
    other = [lv.field_ptr(0, A.LIST_OLD, v) for v in range(24)]
    assert _copy(A, lv, A.LIST_STATE, other, 1) == 0
    s.synchronize()
    assert np.array_equal(np.stack([lv.get_field(0, A.LIST_OLD, v).ravel() for v in range(24)]), got)
    shifted = [lv.field_ptr(0, A.LIST_STATE, max(v - 1, 0)) for v in range(24)]
    assert _copy(A, lv, A.LIST_STATE, shifted, 0) == 0
    s.synchronize()
    assert all(np.array_equal(lv.get_field(0, A.LIST_STATE, v).ravel(), got[0]) for v in range(24))
    lv.close()
