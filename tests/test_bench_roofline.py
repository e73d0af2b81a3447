"""bench.py's rates: the bytes that one launch moves over that launch's time,
however many iterations it advances."""
import importlib.util
import os

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def bench():
    spec = importlib.util.spec_from_file_location("bench", os.path.join(ROOT, "bench.py"))
    mod = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(mod)
    return mod


def test_headline_roofline(bench):
    # 212 iterations of 0.1 ms, four per launch
    r = bench.roofline_of(256 ** 3, 0.1, 0.09, 212, 53, 1.0e9, {"sum2": 6000.0})
    assert r["kernel"] == "fgp_deep3_kernel" and r["iterations_per_launch"] == 4
    assert r["kernel_ms_mean"] == pytest.approx(0.4) and r["kernel_ms_min"] == pytest.approx(0.36)
    assert r["alg_bytes_per_launch"] == 60 * 256 ** 3
    assert r["achieved"] == pytest.approx(60 * 256 ** 3 / 0.4e-3 / 1e9)
    assert r["frac"] == pytest.approx(r["achieved"] / 8000) and r["frac"] < 1
    assert r["frac_of_achievable_sum2"] == pytest.approx(r["achieved"] / 6000)


@pytest.mark.parametrize("kind, n, ms, count, passes", [("pd", 256 ** 3, 0.0733, 50, 17), ("dtv", 256 ** 3, 0.12, 50, 17),
                                                      ("tgv", 192 * 512 * 512, 0.767, 50, 25)])
def test_rates_stay_below_the_peak(bench, kind, n, ms, count, passes):
    r = bench.launch_rate(n, kind, ms, count, passes)
    assert r["kernel_frac_of_8TBps"] < 1
    assert r["kernel_alg_GBps"] * 1e9 * r["launch_ms_mean"] * 1e-3 == pytest.approx(bench.LAUNCH_BYTES[kind] * n)


def test_traffic_file_names_the_kernel_that_runs(bench):
    text = open(bench.TRAFFIC_FILE).read()
    assert "fgp_deep3_kernel" in text and "iterations_per_launch=4" in text
    assert bench.read_traffic(256 ** 3) > 60 * 256 ** 3   # at least what a launch cannot do without
