"""The harness's "auto" tuning can choose what the library does by default:
JACOBI_2D's plan, which no explicit depth and rows give, and SCAN's tiles,
which are not those of 64 doubles per work-item."""

import pytest

from rajaperf_amd.suite import run_suite

pytestmark = pytest.mark.gpu

COMMON = ["--checkrun", "1", "--input-mode", "seeded", "-t", "auto"]


def test_jacobi_auto_takes_the_default_plan(rpx):
    """N = 1002, 40 time steps: four times as fast as any other candidate."""
    res = run_suite(["-k", "Polybench_JACOBI_2D", "--size", "1000000", "--tsteps", "40", *COMMON])
    assert res["rc"] == 0, res.get("failures")
    assert [d["choice"] for d in res["autotune"]] == ["default"]


@pytest.mark.parametrize("choice", ["default", "items_64"])
def test_scan_auto_tells_the_default_from_64_doubles(rpx, tmp_path, choice):
    cache = tmp_path / "tunings"
    args = ["-k", "Algorithm_SCAN", "--size", "1000000", *COMMON, "--tuning-cache", str(cache)]
    assert run_suite(args)["rc"] == 0
    fields = cache.read_text().strip().split("\t")
    cache.write_text("\t".join(fields[:3] + [choice] + fields[4:]) + "\n")
    res = run_suite(args)
    assert res["rc"] == 0, res.get("failures")
    assert [(d["choice"], d["from_cache"]) for d in res["autotune"]] == [(choice, True)]
