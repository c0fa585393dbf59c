"""The reciprocal of the triangular kernels' coefficient sums is the correctly rounded quotient on this hardware: their results are the
oracle's to the bit because of it."""
import ctypes as C
import os

import pytest

pytestmark = pytest.mark.gpu

LIB = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "rocal_amd", "lib", "libreciprocals_check.so")


def test_reciprocal_is_the_quotient():
    import torch
    assert os.path.exists(LIB), "%s is not built (run __graft_entry__.build())" % LIB
    check = C.CDLL(LIB).reciprocals_check
    check.argtypes = [C.c_int, C.c_int, C.c_void_p, C.c_void_p]
    counts = torch.zeros(2, dtype=torch.int64, device="cuda")
    assert check(-40, 40, counts.data_ptr(), torch.cuda.current_stream().cuda_stream) == 0
    assert counts.tolist() == [0, 81 << 23]
