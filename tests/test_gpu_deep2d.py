"""2D passes of many iterations per launch against one iteration per launch.

By default a 2D solve in FP32 arithmetic advances up to eight iterations per
launch with a region of the image in registers (values move between columns by
lane shifts and between row groups through LDS, regions overlap by what the
iterations invalidate, the last pass may be shorter).  Every value is computed
by the one-iteration kernels' expressions, so output and infovector must equal
those of depth=1 (pinned to the oracle by test_gpu_parity.py) bit for bit: at
the edges of the regions (32 and 64 columns, 32 and 64 rows), on thin images,
for partial last passes, every storage type, tolerance stops on any iteration
of a pass, an output buffer that is the input, and values outside the in-range
square roots and divisions (infinities, NaN, zeros, denormals).
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

METHODS = ["rof", "fgp", "pd", "tgv", "dtv", "sb"] + [f"ndf{p}" for p in range(6)]
PRECISION = {"fgp": ["fp32", "bf16", "fp16"], "pd": ["fp32", "bf16", "fp16"], "tgv": ["fp32", "bf16", "fp16"],
             "rof": ["fp32"]}
SHAPES = [(2, 2), (1, 65), (33, 1), (2, 300), (31, 33), (32, 32), (33, 64), (64, 65), (129, 63), (65, 200),
          (300, 257), (1100, 1027)]


def _run(m, x, iters, tol=0.0, nonneg=1, aniso=0, **kw):
    from ccpi.filters import device as D
    if m == "rof":
        return D.rof(x, 0.04, iters, 0.002, tol, **kw)
    if m == "fgp":
        return D.fgp(x, 0.03, iters, tol, aniso, nonneg, **kw)
    if m == "pd":
        return D.pd(x, 0.03, iters, tol, 12.0, aniso, nonneg, **kw)
    if m == "dtv":
        return D.dtv(x, _vol(tuple(x.shape), 99), 0.03, iters, tol, 0.05, aniso, nonneg, **kw)
    if m == "sb":
        return D.sb(x, 0.05, iters, tol, aniso, **kw)
    if m.startswith("ndf"):   # penalty; 0: linear
        return D.ndf(x, 0.3, 0.2 if m != "ndf0" else 0.0, iters, 0.2, int(m[3]) or 1, tol, **kw)
    return D.tgv(x, 0.05, 1.3, 1.7, iters, 12.0, tol, **kw)


def _vol(shape, seed):
    import torch
    g = np.random.default_rng(seed)
    x = g.random(shape).astype(np.float32) * (g.random(shape) > 0.3) - 0.2 * (g.random(shape) > 0.9)
    return torch.from_numpy(x.astype(np.float32)).cuda()


def _bits(t):
    return t.cpu().numpy().view(np.uint32)


def _same(a, b, tag):
    (ya, ia), (yb, ib) = a, b
    assert np.array_equal(ia, ib, equal_nan=True), f"{tag}: infovector {ia} vs {ib}"
    na, nb = ya.isnan(), yb.isnan()
    assert bool((na == nb).all()), f"{tag}: NaN at different places"
    d = (_bits(ya) != _bits(yb)) & ~na.cpu().numpy()
    assert not d.any(), f"{tag}: {int(d.sum())} elements differ"


@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "x".join(map(str, s)))
@pytest.mark.parametrize("method", METHODS)
def test_equal_to_one_iteration_per_launch(method, shape):
    x = _vol(shape, 3)
    for iters in (1, 5, 8, 19):
        for aniso in (0, 1):
            _same(_run(method, x, iters, aniso=aniso, nonneg=aniso, depth=1),
                  _run(method, x, iters, aniso=aniso, nonneg=aniso), f"{method} {shape} iters={iters} aniso={aniso}")
    _same(_run(method, x, 7, depth=1), _run(method, x, 7, depth=2), f"{method} {shape} depth 2")


@pytest.mark.parametrize("method", ["fgp", "pd", "tgv"])
def test_16bit_storage(method):
    x = _vol((150, 190), 4)
    for precision in PRECISION[method][1:]:
        for aniso in (0, 1):
            _same(_run(method, x, 21, aniso=aniso, precision=precision, depth=1),
                  _run(method, x, 21, aniso=aniso, precision=precision), f"{method} {precision} aniso={aniso}")


@pytest.mark.parametrize("check_every", [1, 2, 3, 5])
@pytest.mark.parametrize("method", METHODS)
def test_tolerance_stops(method, check_every):
    x = _vol((120, 140), 5)
    stops = set()
    for tol in (3e-2, 1e-2, 3e-3, 1e-3, 3e-4):
        a = _run(method, x, 90, tol=tol, check_every=check_every, depth=1)
        b = _run(method, x, 90, tol=tol, check_every=check_every)
        _same(a, b, f"{method} tol={tol} check_every={check_every}")
        stops.add(int(a[1][0]))
    if method not in ("ndf1", "ndf5"):   # their flux jumps to +-1: the iterates do not settle
        assert any(k < 90 for k in stops)


@pytest.mark.parametrize("method", METHODS)
def test_output_buffer_is_the_input(method):
    x = _vol((130, 150), 6)
    for tol in (0.0, 1e-3):
        ref = _run(method, x, 30, tol=tol, out=x.clone())
        y = x.clone()
        _same(ref, _run(method, y, 30, tol=tol, out=y), f"{method} tol={tol}")


@pytest.mark.parametrize("method", METHODS)
def test_values_outside_the_fast_ranges(method):
    x = _vol((70, 90), 7)
    x[5:20, 5:20] = 0.0
    x[30:40, :] = 0.5
    x[50, 60] = 1e-39
    x[51, 61] = 3e-33
    x[60, 3] = -1e-35
    for bad in (None, 3e19, 2e38, float("inf"), float("-inf"), float("nan")):
        y = x.clone()
        if bad is not None:
            y[33, 64] = bad
            y[10, 10] = bad
        _same(_run(method, y, 11, nonneg=0, depth=1), _run(method, y, 11, nonneg=0), f"{method} {bad}")


@pytest.mark.parametrize("method", ["fgp", "pd", "tgv", "sb"])
def test_warm_start_across_passes(method):
    from ccpi.filters import device as D
    x = _vol((100, 131), 8)

    def warm(iters, state, ts, cont, **kw):
        if method == "fgp":
            return D.fgp_warm(x, 0.03, iters, state, ts, cont, **kw)
        if method == "pd":
            return D.pd_warm(x, 0.03, iters, state, cont, L=12.0, **kw)
        if method == "sb":
            return D.sb_warm(x, 0.05, iters, state, cont, **kw)
        return D.tgv_warm(x, 0.05, 1.3, 1.7, iters, state, cont, **kw)

    for kw in ({}, {"tol": 2e-3, "check_every": 1}):
        outs = []
        for depth in (1, 0):
            st = D.new_state(method, x)
            st, ts = st if method == "fgp" else (st, None)
            warm(13, st, ts, False, depth=depth, **kw)
            outs.append((warm(22, st, ts, True, depth=depth, **kw), st.clone(), None if ts is None else ts.copy()))
        _same(outs[0][0], outs[1][0], f"{method} {kw}")
        used = [c for c in range(outs[0][1].shape[0]) if bool((outs[0][1][c] != 0).any())]
        for c in used:
            assert bool((outs[0][1][c] == outs[1][1][c]).all()), f"{method} {kw}: state channel {c}"
        if outs[0][2] is not None:
            assert np.array_equal(outs[0][2], outs[1][2])
