"""The kernels' in-range reciprocal and quotient (rcp_in, div_in) against the
device's IEEE division: exact equality, counted on the GPU."""
import ctypes

import pytest

pytestmark = pytest.mark.gpu


def _counts(name, *args, argtypes=()):
    from ccpi.filters.utils import require_gpu_lib
    f = getattr(require_gpu_lib(), name)
    f.argtypes = list(argtypes) + [ctypes.POINTER(ctypes.c_ulonglong)] * 2
    f.restype = ctypes.c_int
    bad, seen = ctypes.c_ulonglong(), ctypes.c_ulonglong()
    assert f(*args, ctypes.byref(bad), ctypes.byref(seen)) == 0
    return bad.value, seen.value


def test_rcp_in_equals_the_ieee_reciprocal_on_every_float_in_range():
    bad, seen = _counts("cilreg_check_rcp_in")
    assert seen == 250 * (1 << 23) + 1   # the floats of [2^-125, 2^125]
    assert bad == 0, f"{bad} floats whose reciprocal is not correctly rounded"


def test_div_in_equals_the_ieee_quotient():
    """Every divisor significand with every 61st dividend significand (the
    offset moves with the divisor), signs and exponents cycling over the range."""
    bad, seen = _counts("cilreg_check_div_in", 61, argtypes=[ctypes.c_uint])
    assert seen > (1 << 46) // 62
    assert bad == 0, f"{bad} quotients that are not correctly rounded"
