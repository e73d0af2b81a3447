"""Edges of the register passes (2D and 3D): values, extents and options at
which a solve could differ from, or be slower than, the kernels it replaced.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _vol(shape, seed):
    import torch
    g = np.random.default_rng(seed)
    return torch.from_numpy((g.random(shape) * (g.random(shape) > 0.3)).astype(np.float32)).cuda()


def _same(a, b, tag):
    import torch
    (ya, ia), (yb, ib) = a, b
    assert np.array_equal(ia, ib, equal_nan=True), f"{tag}: infovector {ia} vs {ib}"
    na, nb = ya.isnan(), yb.isnan()
    assert bool((na == nb).all()), f"{tag}: {int((na != nb).sum())} elements NaN on one side only"
    d = (ya.view(torch.int32) != yb.view(torch.int32)) & ~na
    assert not bool(d.any()), f"{tag}: {int(d.sum())} elements differ"


@pytest.mark.parametrize("precision", ["fp32", "bf16", "fp16"])
@pytest.mark.parametrize("pair", [("inf", "inf"), ("inf", "nan"), ("nan", "-inf"), ("inf", "-inf")], ids=str)
def test_tgv_image_with_adjacent_infinities(pair, precision):
    """Two neighbouring pixels that are infinite or NaN: their dual point holds
    an infinity beside a NaN, which the projection must leave as it is."""
    from ccpi.filters import device as D
    x = _vol((40, 70), 3)
    for y, col, dy, dx in ((5, 6, 0, 1), (20, 33, 0, 1), (31, 62, 0, 1), (12, 50, 1, 0), (31, 20, 1, 0)):
        x[y, col], x[y + dy, col + dx] = float(pair[0]), float(pair[1])
    for iters in (1, 2, 7, 9):
        _same(D.tgv(x, 0.05, 1.3, 1.7, iters, 12.0, precision=precision, depth=1),
              D.tgv(x, 0.05, 1.3, 1.7, iters, 12.0, precision=precision), f"{pair} iters={iters}")


@pytest.mark.parametrize("shape", [(70, 90), (60, 95, 100)], ids=str)
def test_dtv_allocates_once(shape):
    """All of an FGP-dTV solve's memory is one allocation ahead of its first
    kernel: a second one that failed would hand the first back to the pool with
    the reference gradient's kernel still writing it."""
    import ctypes
    from ccpi.filters import device as D
    from ccpi.filters.utils import require_gpu_lib
    lib = require_gpu_lib()
    lib.cilreg_inject_alloc_failure.argtypes = [ctypes.c_int]
    lib.cilreg_inject_alloc_failure.restype = None
    x, ref = _vol(shape, 4), _vol(shape, 5)
    want = D.dtv(x, ref, 0.03, 9, depth=1)
    try:
        lib.cilreg_inject_alloc_failure(1)
        with pytest.raises(RuntimeError, match="alloc"):
            D.dtv(x, ref, 0.03, 9)
        lib.cilreg_inject_alloc_failure(2)   # there is no second allocation to fail
        got = D.dtv(x, ref, 0.03, 9)
    finally:
        lib.cilreg_inject_alloc_failure(0)
    _same(got, want, f"{shape}")
