"""3D passes of several iterations with the pipeline in registers against one
iteration per launch: bit equality of output and infovector over ragged
extents around the regions (64 columns, 16 and 32 rows), thin volumes, chunk
depths down to one plane, partial last passes, every storage type, tolerance
stops on any iteration of a pass, warm starts, an output buffer that is the
input, and values outside the in-range square roots and reciprocals."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# at least half a million voxels each: smaller volumes take other kernels
SHAPES = [(2, 520, 500), (3, 411, 409), (600, 29, 31), (520, 1, 1000), (500, 1010, 1), (90, 64, 90), (61, 97, 130),
          (33, 126, 129), (130, 65, 63)]
METHODS = ["fgp", "pd", "dtv"]
STORED = {"fgp": ["bf16", "fp16"], "pd": ["bf16", "fp16"]}


def _run(m, x, iters, tol=0.0, nonneg=1, aniso=0, **kw):
    from ccpi.filters import device as D
    if m == "pd":
        return D.pd(x, 0.03, iters, tol, 8, aniso, nonneg, **kw)
    if m == "dtv":
        return D.dtv(x, _vol(tuple(x.shape), 99), 0.03, iters, tol, 0.05, aniso, nonneg, **kw)
    return D.fgp(x, 0.03, iters, tol, aniso, nonneg, **kw)


def _vol(shape, seed):
    import torch
    g = np.random.default_rng(seed)
    x = g.random(shape, dtype=np.float32) * (g.random(shape, dtype=np.float32) > 0.3)
    x -= 0.2 * (g.random(shape, dtype=np.float32) > 0.9)
    return torch.from_numpy(x.astype(np.float32)).cuda()


def _same(a, b, tag):
    import torch
    (ya, ia), (yb, ib) = a, b
    assert np.array_equal(ia, ib, equal_nan=True), f"{tag}: infovector {ia} vs {ib}"
    na, nb = ya.isnan(), yb.isnan()
    assert bool((na == nb).all()), f"{tag}: NaN at different places"
    d = (ya.view(torch.int32) != yb.view(torch.int32)) & ~na
    assert not bool(d.any()), f"{tag}: {int(d.sum())} elements differ, first {d.nonzero()[0].tolist()}"


@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "x".join(map(str, s)))
@pytest.mark.parametrize("method", METHODS)
def test_equal_to_one_iteration_per_launch(method, shape):
    x = _vol(shape, 3)
    for iters, aniso in ((1, 0), (4, 1), (11, 0), (6, 1)):
        _same(_run(method, x, iters, aniso=aniso, nonneg=aniso, depth=1),
              _run(method, x, iters, aniso=aniso, nonneg=aniso), f"{method} {shape} iters={iters} aniso={aniso}")
    for zchunk in (1, 3, 17):
        _same(_run(method, x, 5, depth=1), _run(method, x, 5, zchunk=zchunk), f"{method} {shape} zchunk={zchunk}")
    _same(_run(method, x, 7, depth=1), _run(method, x, 7, depth=2), f"{method} {shape} depth 2")


@pytest.mark.parametrize("method", ["fgp", "pd"])
def test_16bit_storage(method):
    x = _vol((70, 90, 100), 4)
    for precision in STORED[method]:
        for aniso in (0, 1):
            _same(_run(method, x, 9, aniso=aniso, precision=precision, depth=1),
                  _run(method, x, 9, aniso=aniso, precision=precision), f"{method} {precision} aniso={aniso}")


@pytest.mark.parametrize("check_every", [1, 2, 3, 5])
@pytest.mark.parametrize("method", METHODS)
def test_tolerance_stops(method, check_every):
    x = _vol((60, 95, 100), 5)
    stops = set()
    for tol in (3e-2, 1e-2, 3e-3, 1e-3):
        a = _run(method, x, 60, tol=tol, check_every=check_every, depth=1)
        b = _run(method, x, 60, tol=tol, check_every=check_every)
        _same(a, b, f"{method} tol={tol} check_every={check_every}")
        stops.add(int(a[1][0]))
    assert any(k < 60 for k in stops)


@pytest.mark.parametrize("method", METHODS)
def test_output_buffer_is_the_input(method):
    x = _vol((62, 90, 95), 6)
    for tol in (0.0, 1e-3):
        ref = _run(method, x, 21, tol=tol, out=x.clone())
        y = x.clone()
        _same(ref, _run(method, y, 21, tol=tol, out=y), f"{method} tol={tol}")


@pytest.mark.parametrize("method", METHODS)
def test_values_outside_the_fast_ranges(method):
    x = _vol((66, 88, 91), 7)
    x[5:20, 5:20, 3:50] = 0.0
    x[30:40] = 0.5
    x[50, 60, 70] = 1e-39
    x[51, 61, 70] = 3e-33
    for bad in (None, 3e19, 2e38, float("inf"), float("nan")):
        y = x.clone()
        if bad is not None:
            y[33, 64, 5] = bad
            y[10, 10, 10] = bad
        _same(_run(method, y, 7, nonneg=0, depth=1), _run(method, y, 7, nonneg=0), f"{method} {bad}")


@pytest.mark.parametrize("method", ["fgp", "pd"])
def test_warm_start_across_passes(method):
    from ccpi.filters import device as D
    x = _vol((60, 91, 97), 8)
    for kw in ({}, {"tol": 2e-3, "check_every": 1}):
        outs = []
        for depth in (1, 0):
            st = D.new_state(method, x)
            st, ts = st if method == "fgp" else (st, None)
            if method == "pd":
                D.pd_warm(x, 0.03, 7, st, False, depth=depth, **kw)
                r = D.pd_warm(x, 0.03, 14, st, True, depth=depth, **kw)
            else:
                D.fgp_warm(x, 0.03, 7, st, ts, False, depth=depth, **kw)
                r = D.fgp_warm(x, 0.03, 14, st, ts, True, depth=depth, **kw)
            outs.append((r, st.clone(), None if ts is None else ts.copy()))
        _same(outs[0][0], outs[1][0], f"{method} {kw}")
        assert bool((outs[0][1] == outs[1][1]).all()), f"{method} {kw}: state"
        assert outs[0][2] is None or np.array_equal(outs[0][2], outs[1][2])
