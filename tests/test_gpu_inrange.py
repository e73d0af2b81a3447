"""The kernels' in-range reciprocal and quotient (rcp_in, div_in) against the
device's IEEE division: exact equality, counted on the GPU."""
import ctypes

import numpy as np
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


@pytest.mark.parametrize("method", ["rof", "llt"])
@pytest.mark.parametrize("shape", [(45, 90), (11, 37, 70)], ids=str)
def test_quotients_below_the_normal_range(method, shape):
    """Tiny differences beside huge ones: the quotients are denormal, some of
    them ties; equal to the oracle bit for bit."""
    import oracle
    import torch
    from ccpi.filters import device as D
    rng = np.random.default_rng(5)
    odd = (2 * rng.integers(0, 8, shape) + 1).astype(np.float32)
    small = rng.integers(-99, -60, shape)
    big = rng.integers(30, 62, shape)
    u = rng.random(shape)
    x = np.where(u < 0.6, np.ldexp(odd, small), np.where(u < 0.9, np.ldexp(odd, big), 0.0)).astype(np.float32)
    ref = oracle.cpu_ref()
    t = torch.from_numpy(x).cuda()
    for iters in (1, 2):
        if method == "rof":
            y, _ = ref.rof(x, 0.02, iters, 1e-3, 0.0)
            z, _ = D.rof(t, 0.02, iters, 1e-3)
        else:
            y, _ = ref.llt(x, 0.01, 0.0085, iters, 1e-4, 0.0)
            z, _ = D.llt(t, 0.01, 0.0085, iters, 1e-4)
        assert np.array_equal(z.cpu().numpy().view(np.int32), np.asarray(y, dtype=np.float32).view(np.int32)), iters
