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


@pytest.mark.parametrize("case", ["dtv image", "dtv volume", "fgp volume on tiles", "tgv volume"])
def test_failure_after_first_kernels_drains(case):
    """A thread's first solve with a tolerance fails to get the pinned block it
    polls through, after kernels that write its device memory were queued: it
    returns with its stream drained, so the memory it hands back to the pool
    is not written any more; the next solve succeeds."""
    import ctypes
    import threading
    import torch
    from ccpi.filters import device as D
    from ccpi.filters.utils import require_gpu_lib
    lib = require_gpu_lib()
    lib.cilreg_inject_alloc_failure.argtypes = [ctypes.c_int]
    lib.cilreg_inject_alloc_failure.restype = None
    x = _vol((70, 90) if "image" in case else (60, 95, 100) if case == "dtv volume" else (20, 33, 67), 4)
    ref = _vol(x.shape, 5)
    big = torch.rand(4096, 4096, device="cuda")

    def run():
        if case.startswith("dtv"):
            return D.dtv(x, ref, 0.03, 9, 1e-9)
        return D.fgp(x, 0.03, 9, 1e-9) if case.startswith("fgp") else D.tgv(x, 0.03, 1.0, 2.0, 9, 12.0, 1e-9)

    want = run()
    torch.mm(big, big)
    torch.cuda.synchronize()
    res = {}

    def first_of_a_thread():
        s = torch.cuda.Stream()
        with torch.cuda.stream(s):
            for _ in range(60):
                torch.mm(big, big)
            res["busy"] = not s.query()
            lib.cilreg_inject_alloc_failure(2)   # after the solve's device memory
            try:
                run()
            except RuntimeError as e:
                res["error"] = str(e)
            finally:
                lib.cilreg_inject_alloc_failure(0)
            res["drained"] = s.query()
            res["again"] = run()

    t = threading.Thread(target=first_of_a_thread)
    t.start()
    t.join()
    torch.cuda.synchronize()
    assert res["busy"]
    assert "alloc" in res.get("error", ""), res.get("error", "no error")
    assert res["drained"], "the failed solve left work on its stream"
    _same(res["again"], want, case)


@pytest.mark.parametrize("rows", [1, 2, 3, 4, 5, 7, 8, 9])
@pytest.mark.parametrize("method", ["fgp", "pd", "tgv", "rof", "sb", "ndf", "dtv"])
def test_images_of_few_rows(method, rows):
    """Long images that regions of 4 and 8 rows cover, and one row more: equal
    to one iteration per launch in every storage type, with and without stops,
    at widths around one and several regions."""
    from ccpi.filters import device as D

    def run(x, iters, tol, p, **kw):
        if method == "fgp":
            return D.fgp(x, 0.03, iters, tol, 0, 1, precision=p, **kw)
        if method == "pd":
            return D.pd(x, 0.03, iters, tol, 8, 1, 1, precision=p, **kw)
        if method == "tgv":
            return D.tgv(x, 0.05, 1.3, 1.7, iters, 12.0, tol, precision=p, **kw)
        if method == "rof":
            return D.rof(x, 0.04, iters, 0.002, tol, **kw)
        if method == "sb":
            return D.sb(x, 0.05, iters, tol, 0, **kw)
        if method == "ndf":
            return D.ndf(x, 0.3, 0.2, iters, 0.2, 2, tol, **kw)
        return D.dtv(x, _vol(tuple(x.shape), 9), 0.03, iters, tol, 0.05, 0, 1, **kw)

    for width in (63, 64, 65, 40011):
        x = _vol((rows, width), rows)
        for p in ("fp32", "bf16", "fp16") if method in ("fgp", "pd", "tgv") else ("fp32",):
            for iters, tol in ((19, 0.0), (25, 2e-2)):
                kw = {"check_every": 2} if tol else {}
                _same(run(x, iters, tol, p, depth=1, **kw), run(x, iters, tol, p, **kw),
                      f"{method} {rows} x {width} {p} tol={tol}")


@pytest.mark.parametrize("shape", [(1, 1), (1, 2), (2, 1), (1, 40), (1, 63), (1, 500), (31, 1), (33, 1), (64, 1), (65, 1),
                                   (700, 1), (1, 30011), (30011, 1)], ids=str)
def test_rof_on_a_single_row_or_column(shape):
    """The mirrored neighbour of a single column or row is the point itself."""
    from ccpi.filters import device as D
    x = _vol(shape, 6)
    for iters, tol in ((1, 0.0), (8, 0.0), (43, 0.0), (60, 1e-3)):
        _same(D.rof(x, 0.04, iters, 0.002, tol, depth=1, check_every=3), D.rof(x, 0.04, iters, 0.002, tol, check_every=3),
              f"{shape} iters={iters} tol={tol}")


@pytest.mark.parametrize("shape", [(140, 2, 2000), (90, 3, 2000), (70, 4, 2000), (60, 5, 1900), (24000, 3, 9), (2, 520, 500),
                                   (2, 2048, 2048), (3, 420, 410), (3, 1500, 1400), (4, 360, 365), (5, 1120, 1000),
                                   (103, 56, 125), (128, 48, 128), (256, 8, 512)], ids=lambda s: "x".join(map(str, s)))
@pytest.mark.parametrize("method", ["fgp", "pd", "dtv"])
def test_volumes_of_few_rows_or_planes(method, shape):
    """Extents on either side of the lines between the register and the tiled
    passes: equal to one iteration per launch in every storage type, with and
    without checks."""
    from ccpi.filters import device as D

    def run(tol, p, **kw):
        if method == "dtv":
            return D.dtv(x, ref, 0.03, 7, tol, 0.05, 0, 1, **kw)
        return (D.fgp if method == "fgp" else D.pd)(x, 0.03, 7, tol, *((8,) if method == "pd" else ()), 0, 1,
                                                     precision=p, **kw)

    x, ref = _vol(shape, 2), _vol(shape, 8)
    for p in ("fp32", "bf16", "fp16") if method != "dtv" else ("fp32",):
        for tol in (0.0, 1e-9):
            kw = {"check_every": 2} if tol else {}
            _same(run(tol, p, depth=1, **kw), run(tol, p, **kw), f"{method} {shape} {p} tol={tol}")


@pytest.mark.parametrize("method", ["rof", "fgp", "pd", "tgv"])
def test_applying_an_images_tuned_choice_is_the_default(method):
    """The options that autotune returns for an image, handed to the solve, give
    the default's kernels: the fastest pass is as fast (one iteration per launch
    takes more than twice as long), and the results are the same."""
    from ccpi.filters import device as D
    x = _vol((512, 512), 7)
    c = D.autotune(method, (512, 512))

    def run(**kw):
        if method == "rof":
            r = D.rof(x, 0.04, 160, 0.002, profile=True, **kw)
        elif method == "tgv":
            r = D.tgv(x, 0.05, 1.3, 1.7, 160, 12.0, profile=True, **kw)
        else:
            r = (D.fgp if method == "fgp" else D.pd)(x, 0.03, 160, profile=True, **kw)
        return r, D.last_profile()[1]

    tuned = {k: c[k] for k in ("tile_y", "zchunk", "depth")}
    run()
    (a, ta), (b, tb), (_, t1) = run(), run(**tuned), run(depth=1)
    _same(a, b, method)
    assert tb < 0.5 * (ta + t1), f"us per iteration: default {1e3 * ta}, tuned {1e3 * tb}, one per launch {1e3 * t1}"


@pytest.mark.parametrize("method", ["fgp", "pd"])
def test_tuner_times_the_middle_of_a_register_solve(method):
    """On a volume the register passes take, a probe holds several of them: four
    iterations were one pass that read no state and wrote none.  The choice is
    one of the candidates and leaves the results alone."""
    from ccpi.filters import device as D
    shape = (70, 90, 110)
    D.tune_clear()
    c = D.autotune(method, shape)
    assert D.last_profile()[2] == 16
    assert c["tile_y"] in (4, 8) and c["zchunk"] in (0, 8, 16, 32) and c["depth"] in (1, 2) and c["ms_per_iter"] > 0
    x = _vol(shape, 3)
    f = D.fgp if method == "fgp" else D.pd
    _same(f(x, 0.03, 9, tile_y=c["tile_y"], zchunk=c["zchunk"], depth=c["depth"]), f(x, 0.03, 9), method)


@pytest.mark.parametrize("method", ["fgp", "pd"])
def test_tuner_times_a_groups_own_passes(method, tmp_path):
    """The probe for a grouped job runs the tiled passes that the group runs: two
    iterations each at depth 2, also where a single solve of the stacked extent
    would run in registers."""
    import ctypes
    from ccpi.filters import batch as B, device as D
    from ccpi.filters.utils import require_gpu_lib
    lib = require_gpu_lib()
    lib.cilreg_last_profile_passes.restype = ctypes.c_int
    D.tune_clear()
    x = _vol((40, 70, 100), 1)
    spec = {"method": method, "input": x, "iters": 6, "lambda": 0.03, "L": 12.0}
    B.batch_run([spec, dict(spec)], autotune=True)
    D.tune_save(tmp_path / "t.txt")
    rows = [l.split() for l in open(tmp_path / "t.txt") if not l.startswith("#")]
    assert len(rows) == 1 and rows[0][4] == "1"   # the grouped entry
    depth = int(rows[0][10])
    assert D.last_profile()[2] == 8 and lib.cilreg_last_profile_passes() == 8 // depth


def test_choices_timed_on_earlier_kernels_are_not_used(tmp_path):
    """An entry for this device without the kernels' generation was timed before
    the register passes: it loads and saves, and the tuner times anew."""
    from ccpi.filters import device as D
    shape = (70, 90, 110)
    D.tune_clear()
    D.autotune("fgp", shape)
    D.tune_save(tmp_path / "new.txt")
    header, row = [l for l in open(tmp_path / "new.txt") if not l.startswith("# device")]
    f = row.split()
    assert f[0].count(":") == 2
    f[0] = f[0].rsplit(":", 1)[0]
    f[8:11] = ["4", "8", "1"]
    f[11] = "123.0"
    (tmp_path / "old.txt").write_text(header + " ".join(f) + "\n")
    D.tune_clear()
    assert D.tune_load(tmp_path / "old.txt") == 1
    assert D.autotune("fgp", shape)["ms_per_iter"] != 123.0
    assert D.tune_entries() == 2   # the old entry is still there to save
    D.tune_clear()


@pytest.mark.parametrize("precision", ["fp32", "bf16"])
@pytest.mark.parametrize("shape, in_place", [((1100, 1000), True), ((1300, 1380), True), ((1401, 1301), False)], ids=str)
def test_allocation_free_large_image_two_iterations_per_launch(shape, in_place, precision):
    """depth=2 on an image of 2^20 pixels and more: two iterations per launch in a
    workspace of eight fields (nine in place); ten were reserved for passes of
    one iteration, which left no room from 1.68 million pixels on."""
    import ctypes
    import torch
    from ccpi.filters import device as D
    from ccpi.filters.utils import last_error, require_gpu_lib
    f = require_gpu_lib().cilreg_fgp_dev_noalloc
    vp, i, fl = ctypes.c_void_p, ctypes.c_int, ctypes.c_float
    f.argtypes, f.restype = [vp, vp, vp, fl, i, fl, i, i, i, i, i, vp, vp], i
    for iters in (1, 2, 7):
        x = _vol(shape, 5)
        want = D.fgp(x, 0.03, iters, 0.0, 0, 1, precision=precision, depth=1)
        out = x if in_place else torch.zeros_like(x)
        info = np.zeros(2, dtype=np.float32)
        opts = D.make_opts(precision=precision, depth=2)
        rc = f(x.data_ptr(), out.data_ptr(), info.ctypes.data, 0.03, iters, 0.0, 0, 1, shape[1], shape[0], 1,
               ctypes.byref(opts), ctypes.c_void_p(torch.cuda.current_stream().cuda_stream))
        assert rc == 0, last_error()
        _same((out, info), want, f"{shape} iters={iters}")


def _same64(a, b, tag):
    import torch
    assert np.array_equal(a[1], b[1]), f"{tag}: infovector {a[1]} vs {b[1]}"
    assert bool((a[0].view(torch.int64) == b[0].view(torch.int64)).all()), tag


@pytest.mark.parametrize("wide_index", [False, True])
@pytest.mark.parametrize("tile_y", [4, 8])
def test_fp64_images_two_iterations_per_pass(tile_y, wide_index):
    """The two-iteration tiled pass of an image, which only FP64 still takes:
    equal to one iteration per launch on both tile heights with either index
    width, for odd and even counts and stops on either iteration of a pass."""
    from ccpi.filters import device as D
    kw = dict(tile_y=tile_y, wide_index=wide_index)
    for shape in ((5, 7), (33, 64), (63, 65), (130, 201)):
        x = _vol(shape, 3).double()
        for iters, aniso in ((1, 0), (2, 1), (9, 0), (10, 1)):
            _same64(D.fgp_f64(x, 0.03, iters, 0.0, aniso, 1, depth=1, **kw),
                    D.fgp_f64(x, 0.03, iters, 0.0, aniso, 1, depth=2, **kw), f"{shape} iters={iters}")
    stops = set()
    x = _vol((120, 140), 5).double()
    for check_every in (1, 2, 3):
        for tol in (3e-2, 2e-2, 1e-2, 5e-3, 3e-3):
            a = D.fgp_f64(x, 0.03, 90, tol, 0, 1, depth=1, check_every=check_every, **kw)
            _same64(a, D.fgp_f64(x, 0.03, 90, tol, 0, 1, depth=2, check_every=check_every, **kw),
                    f"tol={tol} check_every={check_every}")
            stops.add(int(a[1][0]))
    assert {k & 1 for k in stops if k < 90} == {0, 1}


@pytest.mark.parametrize("method", ["rof", "fgp", "pd", "tgv", "dtv", "sb", "ndf"])
def test_one_iteration_kernels_of_images_with_64_bit_indexes(method):
    """depth=1 keeps the one-iteration kernels; both index widths agree."""
    from ccpi.filters import device as D
    x, ref = _vol((101, 133), 3), _vol((101, 133), 4)

    def run(**kw):
        if method == "rof":
            return D.rof(x, 0.04, 13, 0.002, 1e-9, depth=1, **kw)
        if method == "fgp":
            return D.fgp(x, 0.03, 13, 1e-9, 0, 1, depth=1, **kw)
        if method == "pd":
            return D.pd(x, 0.03, 13, 1e-9, 12.0, 0, 1, depth=1, **kw)
        if method == "tgv":
            return D.tgv(x, 0.05, 1.3, 1.7, 13, 12.0, 1e-9, depth=1, **kw)
        if method == "dtv":
            return D.dtv(x, ref, 0.03, 13, 1e-9, 0.05, 0, 1, depth=1, **kw)
        if method == "sb":
            return D.sb(x, 0.05, 13, 1e-9, 0, depth=1, **kw)
        return D.ndf(x, 0.3, 0.2, 13, 0.2, 2, 1e-9, depth=1, **kw)

    _same(run(), run(wide_index=True), method)


@pytest.mark.parametrize("precision", ["bf16", "fp16"])
def test_tgv_16bit_one_iteration_kernel_with_64_bit_indexes(precision):
    from ccpi.filters import batch as B, device as D
    x = _vol((13, 37, 70), 3)
    want = D.tgv(x, 0.05, 1.3, 1.7, 9, 12.0, 1e-9, precision=precision, depth=1)
    _same(want, D.tgv(x, 0.05, 1.3, 1.7, 9, 12.0, 1e-9, precision=precision, depth=1, wide_index=True), precision)
    spec = {"method": "tgv", "input": x, "iters": 9, "lambda": 0.05, "alpha1": 1.3, "alpha0": 1.7, "L2": 12.0}
    (y, _), = B.batch_run([spec], precision=precision, depth=1, wide_index=True)
    assert bool((y == want[0]).all())
