"""Host side of the field copies: the comparison that finds edits in large
arrays, whatever chunk the difference lies in."""
import ctypes as C

import numpy as np
import pytest

from akantu2_amd import _native as N
from akantu2_amd.model import _LARGE, _Mirror

CHUNK = 1 << 20


@pytest.mark.parametrize("n", [0, 1, CHUNK - 1, CHUNK, 5 * CHUNK + 3, 40 * CHUNK])
def test_host_differs(n):
    a = np.random.default_rng(0).integers(0, 255, n, dtype=np.uint8)
    b = a.copy()

    def differs():
        d = C.c_int(-1)
        N.check(N.lib().akx_host_differs(a.ctypes.data_as(C.c_void_p),
                                         b.ctypes.data_as(C.c_void_p), n, C.byref(d)))
        return d.value

    if n:
        assert differs() == 0
    for at in {0, n // 2, n - 1, CHUNK, 3 * CHUNK - 1}:
        if 0 <= at < n:
            b[at] ^= 1
            assert differs() == 1
            b[at] ^= 1


def test_large_mirror_sees_an_edit():
    mir = _Mirror(np.zeros((_LARGE // 24 + 7, 3)), True)
    assert not mir.edited()
    mir.base[-1, 2] = -0.0  # another bit pattern of zero is an edit too
    assert mir.edited()
