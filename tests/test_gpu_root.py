"""GPU check that the pair terms' quotient by a root (div_root in
pbf-cuda_amd/csrc/pbf_device.h), whose reciprocal starts from the root's own
estimate, is div_pair's for every root of a positive float from 2^-90 to 2^10:
it divides by the same reciprocal bit for bit, or, at the roots where the two
estimates lead to different ones, its quotients by all numerators are the IEEE
quotients (test_gpu_arith checks the root and div_pair)."""
import ctypes

import pytest

from test_gpu_arith import LIB, _bits

pytestmark = pytest.mark.gpu


def test_quotient_by_a_root_is_ieee(device):
    import torch  # noqa: F401  (the HIP runtime torch loaded)

    fn = ctypes.CDLL(LIB).pbf_check_root_quotient
    fn.argtypes = [ctypes.c_uint32, ctypes.c_uint32, ctypes.c_ulonglong * 2]
    fn.restype = ctypes.c_int
    out = (ctypes.c_ulonglong * 2)(1, 1)
    assert fn(_bits(2.0 ** -90), _bits(2.0 ** 10), out) == 0
    print(f"other reciprocals {out[0]}, wrong quotients by them {out[1]}", flush=True)
    assert out[0] <= 4096  # all of them listed and swept
    assert out[1] == 0
