"""lmie_amd.abi reads output blocks through pointers of the C library (CPU)."""
import ctypes as C

import numpy as np
import pytest

from lmie_amd import abi


@pytest.mark.parametrize("shape", [(1,), (16,), (17,), (6, 64)])
def test_a_missing_block_raises(shape):
    """Short and long blocks alike: an exception, not a read through NULL."""
    with pytest.raises(ValueError):
        abi._arr(C.POINTER(C.c_double)(), shape)


@pytest.mark.parametrize("shape", [(0,), (6, 0), (1,), (16,), (17,), (6, 64)])
def test_blocks_are_copied(shape):
    src = np.arange(np.prod(shape), dtype=float).reshape(shape)
    got = abi._arr(src.ctypes.data_as(C.POINTER(C.c_double)), shape)
    assert np.array_equal(got, src) and got.shape == shape
    got += 1.0
    assert src.size == 0 or src.flat[0] == 0.0
