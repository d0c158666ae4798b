"""How a step's lists become the library's arrays (tq_kv_amd/engine/engine.py, tq_kv_amd/native.py): on the host alone."""
import ctypes

import numpy as np
import pytest
import torch

from tq_kv_amd import native
from tq_kv_amd.engine.engine import _int32


@pytest.mark.parametrize("values", [
    [], [0], [5, 0, 2 ** 31 - 1], [2 ** 31], [2 ** 63 - 1, 3], [-1, -2, -2 ** 31], [-2 ** 31 - 1, 7], [np.int64(2 ** 40), 1], [np.int32(4), True], list(range(3000))])
def test_numbers_of_more_than_32_bits_stay_outside_of_every_range(values):
    got = _int32(values)
    assert got.dtype == np.int32 and got.flags["C_CONTIGUOUS"]
    assert got.tolist() == np.asarray(values, dtype=np.int64).clip(-1, 2 ** 31 - 1).tolist()


# (elements with dimensions, and 0-d arrays, are cast by numpy and not looked at one by one)
@pytest.mark.parametrize("many", [[np.array([2 ** 32 + 3]), np.array([4])], [np.array(2 ** 32 + 3)], [np.array(-2 ** 32 + 3), 5], [torch.tensor(2 ** 32 + 3), torch.tensor(7)],
                                  list(torch.tensor([[2 ** 32 + 3], [4]])), [[2 ** 32 + 3, 1], [2, 3]], np.array([2 ** 32 + 5, 6]), torch.tensor([2 ** 32 + 5, 6]),
                                  [np.uint32(2 ** 32 - 1)], [3e9, 1.5], [True, np.int16(-7)], (2 ** 31, 2), np.array([-9, 4], dtype=np.int32)])
def test_numbers_in_arrays_and_tensors_stay_outside_of_every_range_too(many):
    before = many.copy() if isinstance(many, np.ndarray) else None
    got = _int32(many)
    want = np.asarray(many, dtype=np.int64).clip(-1, 2 ** 31 - 1)
    assert got.dtype == np.int32 and got.flags["C_CONTIGUOUS"] and got.shape == want.shape and got.tolist() == want.tolist()
    assert before is None or (many == before).all()


def test_an_array_is_passed_by_its_own_memory():
    whole = np.arange(8, dtype=np.int32)
    fixed = whole.copy()
    fixed.flags.writeable = False
    for a in (whole, whole[2:], whole[:0], fixed):
        p = native._ptr(a)
        assert isinstance(p, native._I32P) and [p[i] for i in range(a.size)] == a.tolist()
        assert a.size == 0 or ctypes.addressof(p.contents) == a.ctypes.data
    assert native._ptr(None) is None
