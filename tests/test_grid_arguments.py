"""mo_grid_build refuses a resolution out of range by its argument, before
any device memory is asked for (its workspace grows with the number of
bricks).  The pointers are never followed."""
import ctypes as C

import numpy as np
import pytest

from meshode_amd import _lib


@pytest.mark.parametrize("N", [1, 0, -5, -100000, 2049, 5000, 100000, 2 ** 31 - 1])
def test_grid_resolution_out_of_range(N):
    V, F = np.zeros((3, 3)), np.array([[0, 1, 2]], np.int32)
    with pytest.raises(_lib.MoError, match=rf"grid resolution {N} out of range"):
        _lib.call("mo_grid_build", C.c_void_p(V.ctypes.data), 3, C.c_void_p(F.ctypes.data), 1, N, C.c_void_p(0),
                  C.c_void_p(0), C.c_void_p(0), C.c_void_p(0))
