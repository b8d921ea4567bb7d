"""The softcaps that leave out cases which cannot occur in their range
(gemmaedge_amd/csrc/ge_math.h, softcap_range) against the general one, on the
GPU, for every float of the range: bit-identical but for the sign of zero."""
import ctypes
import os

import pytest

pytestmark = pytest.mark.gpu

LIB = os.path.join(os.path.dirname(os.path.abspath(__file__)), "cpp", "lib", "libge_math_check.so")


@pytest.mark.parametrize("cap", [30.0, 50.0, 5.0, 1.0, 0.3, 7.0e5, 23.7])
@pytest.mark.parametrize("which", [1, 2])
def test_softcap_range_equals_softcap(which, cap):
    import torch

    assert torch.cuda.is_available(), "GPU test run without a GPU"
    lib = ctypes.CDLL(LIB)
    lib.ge_test_softcap_range_mismatches.restype = ctypes.c_longlong
    lib.ge_test_softcap_range_mismatches.argtypes = [ctypes.c_int, ctypes.c_float]
    print(f"[softcap] range {which} cap {cap}", flush=True)
    assert lib.ge_test_softcap_range_mismatches(which, cap) == 0
