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


@pytest.mark.parametrize("dtype,refused", [(np.float32, (ctypes.c_int, ctypes.c_double)), (np.int32, (ctypes.c_float, ctypes.c_double)),
                                           (np.float64, (ctypes.c_float, ctypes.c_int))])
@pytest.mark.parametrize("shape", [(0, 4), (1, 4), (3, 4)])
def test_pointers_have_their_type(dtype, refused, shape):
    """A prototype with a typed pointer takes what _pointer and _row_pointers give for its type and refuses that of others, as it
    refuses numbers."""
    x = np.zeros(shape, dtype)
    own = cb._C_TYPES[np.dtype(dtype).char][0]
    ctypes.POINTER(own).from_param(cb._pointer(x))
    ctypes.POINTER(ctypes.POINTER(own)).from_param(cb._row_pointers(x))
    for other in refused:
        with pytest.raises(TypeError):
            ctypes.POINTER(other).from_param(cb._pointer(x))
        with pytest.raises(TypeError):
            ctypes.POINTER(ctypes.POINTER(other)).from_param(cb._row_pointers(x))


def test_library_calls_refuse_pointers_of_another_type():
    lib = cb.load_library()
    x = np.zeros((2, 3), np.float32)
    handle = lib.ModelCalcerCreate()
    try:
        for rows, out in ((cb._row_pointers(x.astype(np.int32)), cb._pointer(np.zeros(2))), (cb._row_pointers(x), cb._pointer(x)),
                          (cb._row_pointers(x), x.ctypes.data), (x.ctypes.data, cb._pointer(np.zeros(2)))):
            with pytest.raises(ctypes.ArgumentError):
                lib.CalcModelPredictionFlat(handle, 2, rows, 3, out, 2)
    finally:
        lib.ModelCalcerDelete(handle)


def test_rows_at_addresses_beyond_what_a_signed_number_holds(monkeypatch):
    x = np.zeros((3, 4), np.float32)
    monkeypatch.setattr(cb, "_address", lambda a: (1 << 63) + 64)
    argument = cb._row_pointers(x)
    rows = ctypes.cast(argument, ctypes.POINTER(ctypes.c_void_p))
    assert [rows[i] for i in range(3)] == [(1 << 63) + 64 + 16 * i for i in range(3)]
