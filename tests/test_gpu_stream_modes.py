"""COPY, MUL, ADD and TRIAD around the length where their accesses turn
nontemporal, by default and with either kind asked for, against numpy, bit for
bit; and the harness's tunings of both kinds."""

import numpy as np
import pytest

from rajaperf_amd.suite import run_suite

pytestmark = pytest.mark.gpu

FROM = 15 << 19   # two inputs
FROM1 = 12 << 20  # one


@pytest.mark.parametrize("n", [1, 513, 100_003, FROM - 1, FROM, FROM + 1, FROM1 - 1, FROM1])
def test_streams_in_every_mode(rpx, rng, n):
    L = rpx.lib()
    a, b = rng.random(n), rng.random(n)
    da, db, out = rpx.DeviceBuffer.from_array(a), rpx.DeviceBuffer.from_array(b), rpx.DeviceBuffer(8 * n)
    calls = [(lambda t: L.rpx_copy_f64(out.ptr, da.ptr, n, t, None), a),
             (lambda t: L.rpx_mul_f64(out.ptr, da.ptr, 0.75, n, t, None), 0.75 * a),
             (lambda t: L.rpx_add_f64(out.ptr, da.ptr, db.ptr, n, t, None), a + b),
             (lambda t: L.rpx_triad_f64(out.ptr, da.ptr, db.ptr, 0.75, n, t, None), a + 0.75 * b)]
    for flags in (None, rpx.RPX_TUNE_CACHED, rpx.RPX_TUNE_NONTEMPORAL,
                  rpx.RPX_TUNE_CACHED | rpx.RPX_TUNE_NONTEMPORAL):
        for call, want in calls:
            L.rpx_fill_const_f64(out.ptr, n, -1.0, None)
            call(None if flags is None else rpx.tuning(flags=flags))
            assert np.array_equal(out.to_array(), want)


def test_harness_offers_both(rpx):
    res = run_suite(["-k", "Stream_TRIAD", "--size", "1000", "--checkrun", "1", "-t", "cached", "nontemporal"])
    assert res["rc"] == 0, res.get("failures")
    assert [r["tuning"] for r in res["runs"]] == ["cached", "nontemporal"]
