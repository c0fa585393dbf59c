"""The addresses under which the op classes hand parameter arrays to the C library: those of the array that is kept alive for the call,
whatever form the caller's values come in."""
import numpy as np
import pytest

from rocal_amd import ops


def _read_only(a):
    a = a.copy()
    a.flags.writeable = False
    return a


@pytest.mark.parametrize("make", [
    lambda a: a,
    _read_only,
    lambda a: a.tolist(),
    lambda a: a.astype(np.int64),
    lambda a: np.asfortranarray(a),
    lambda a: np.repeat(a, 2, axis=0)[::2],
    lambda a: np.broadcast_to(a, a.shape),
    lambda a: a.view(np.recarray),
    lambda a: a.reshape(-1)[:0],
], ids=["as is", "read-only", "list", "other type", "column order", "strided", "broadcast", "subclass", "empty"])
def test_address_is_that_of_the_kept_array(make):
    values = make(np.arange(12, dtype=np.uint32).reshape(3, 4))
    kept, address = ops._arr(values, np.uint32)
    assert kept.dtype == np.uint32 and kept.flags.c_contiguous and np.array_equal(kept, np.asarray(values))
    assert address == kept.ctypes.data
    if isinstance(values, np.ndarray) and values.dtype == np.uint32 and values.flags.c_contiguous:
        assert np.shares_memory(kept, values) or values.size == 0  # (an array in the right form is handed over as it is)


def test_no_array_is_no_address():
    assert ops._arr(None, np.float32) == (None, None)
