"""Addresses that the Python calls hand to the library: of rows of any number and kind of memory."""
import ctypes

import numpy as np
import pytest

import catboost_amd as cb


@pytest.mark.parametrize("shape,kind", [
    ((0, 4), "plain"), ((1, 4), "plain"), ((2, 4), "plain"), ((3, 0), "plain"), ((257, 1), "plain"), ((1, 4), "read-only"),
    ((5, 3), "read-only"), ((4, 3), "view"),
])
def test_row_pointers(shape, kind):
    x = np.arange(shape[0] * shape[1], dtype=np.float32).reshape(shape)
    if kind == "view":
        x = np.concatenate([x, x])[2:2 + shape[0]]
    x.setflags(write=kind != "read-only")
    assert cb._address(x) == x.ctypes.data
    argument = cb._row_pointers(x)  # owns the addresses; a cast of it does not
    rows = ctypes.cast(argument, ctypes.POINTER(ctypes.c_void_p))
    for i in range(shape[0]):
        assert rows[i] == x.ctypes.data + i * x.strides[0]
        if shape[1]:
            assert ctypes.cast(rows[i], ctypes.POINTER(ctypes.c_float))[0] == x[i, 0]
