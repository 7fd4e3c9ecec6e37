"""Host result arrays: shapes, types, addresses in the order of the C struct, and
memory of their own (keeping one array of a call keeps no other alive)."""
import ctypes as C

import numpy as np
import pytest

from qmcbeaver_amd._abi import ResultArrays, Results


@pytest.mark.parametrize("num,N", [(0, 4), (1, 1), (7, 5), (256, 64)])
def test_arrays_and_addresses(num, N):
    r = ResultArrays(num, N)
    assert tuple(f for f, _ in Results._fields_) == ResultArrays.FIELDS
    for f in ResultArrays.FIELDS:
        a = r[f]
        shape = {"grad_lnpsi": (num, N, 3), "mod_drift": (num, N, 3), "r2": (num, 3)}.get(f, (num,))
        assert a.shape == shape and a.flags.c_contiguous and not a.any()
        assert a.dtype == (np.int8 if f in ("sign_psi", "singular") else np.float64)
        assert C.cast(getattr(r.struct, f), C.c_void_p).value == a.ctypes.data
        assert a.base is None  # owns its memory
