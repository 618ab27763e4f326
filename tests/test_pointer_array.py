"""The C pointer array of a call, from every kind of sequence that callers pass."""

import ctypes

import numpy as np
import pytest

from elasticmegatron_amd._native import _ptr_array

VALUES = [0, 16, 2 ** 47 - 16, 2 ** 63 + 32, 2 ** 64 - 16]


@pytest.mark.parametrize("n", [1, 2, 5, 900])
@pytest.mark.parametrize("kind", [list, tuple, lambda v: np.array(v, dtype=np.uint64),
                                  lambda v: [np.uint64(x) for x in v]], ids=["list", "tuple", "numpy", "scalars"])
def test_values(n, kind):
    v = (VALUES * n)[:n]
    a = _ptr_array(kind(v))
    assert len(a) == n and [a[i] or 0 for i in range(n)] == v
    assert ctypes.sizeof(a) == 8 * n


def test_empty_and_refused():
    assert len(_ptr_array([])) == 1 and not _ptr_array([])[0]
    for bad in ([-1], [2 ** 64], [None], [[1, 2]]):
        with pytest.raises((OverflowError, TypeError, ValueError)):
            _ptr_array(bad)
    assert _ptr_array([16.0])[0] == 16   # numpy's conversion, as for a tuple
