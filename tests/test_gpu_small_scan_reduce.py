"""SCAN, DOT and REDUCE_SUM at the sizes where their default shapes change, in
turn on one scratch each, exact on integers; and with a scratch that only the
large-array layouts fit."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SIZES = [1, 2, 4095, 4096, 4097, 8193, (1 << 20) + 1, 1 << 20, 5, (1 << 21) + 3, 1 << 21, (1 << 22) + 1, 1 << 22, 4096,
         (1 << 23) + 1, 1 << 23]


def test_one_scratch_for_all_sizes(rpx, rng):
    L, top = rpx.lib(), max(SIZES)
    x, w = rng.integers(-9, 10, top).astype(float), rng.integers(-9, 10, top).astype(float)
    dx, dw, y, res = rpx.DeviceBuffer.from_array(x), rpx.DeviceBuffer.from_array(w), rpx.DeviceBuffer(8 * top), \
        rpx.DeviceBuffer(8)
    reduces, scans = ([f(n, None) for n in sorted(SIZES)]
                      for f in (L.rpx_reduce_scratch_bytes, L.rpx_scan_scratch_bytes))
    assert reduces == sorted(reduces) and scans == sorted(scans)
    rb, sb = reduces[-1], scans[-1]
    red, scr = rpx.DeviceBuffer(rb), rpx.DeviceBuffer(sb)
    L.rpx_reduce_scratch_init(red.ptr, rb, None)
    L.rpx_scan_scratch_init(scr.ptr, sb, None)
    for n in SIZES * 2:
        print(n, flush=True)
        L.rpx_dot_f64(dx.ptr, dw.ptr, n, res.ptr, 0, red.ptr, rb, None, None)
        L.rpx_dot_f64(dx.ptr, dw.ptr, n, res.ptr, 1, red.ptr, rb, None, None)
        assert res.to_array()[0] == 2 * np.dot(x[:n], w[:n])
        L.rpx_reduce_sum_f64(dx.ptr, n, res.ptr, red.ptr, rb, None, None)
        assert res.to_array()[0] == x[:n].sum()
        for scan, ref in ((L.rpx_scan_exclusive_f64, np.r_[0, np.cumsum(x[:n])[:-1]]),
                          (L.rpx_scan_inclusive_f64, np.cumsum(x[:n]))):
            scan(dx.ptr, y.ptr, n, scr.ptr, sb, None, None)
            assert np.array_equal(y.to_array()[:n], ref)
    assert not red.to_array().any()
    assert L.rpx_scan_scratch_status(scr.ptr) == 0


@pytest.mark.parametrize("n", [50001, (1 << 20) - 1])
def test_scratch_of_the_large_layouts(rpx, rng, n):
    L = rpx.lib()
    x = rng.integers(-9, 10, n).astype(float)
    dx, y, res = rpx.DeviceBuffer.from_array(x), rpx.DeviceBuffer(8 * n), rpx.DeviceBuffer(8)
    rb = L.rpx_reduce_scratch_bytes(n, rpx.tuning(512, 32))  # the tickets' layout
    sb = 256 + 3 * -(-(8 * -(-n // 16384)) // 256) * 256     # words of 16384-element tiles
    assert rb < L.rpx_reduce_scratch_bytes(n, None) or n < (1 << 18)
    assert sb < L.rpx_scan_scratch_bytes(n, None) or n < (1 << 18)
    red, scr = rpx.DeviceBuffer(rb), rpx.DeviceBuffer(sb)
    L.rpx_reduce_scratch_init(red.ptr, rb, None)
    L.rpx_scan_scratch_init(scr.ptr, sb, None)
    for _ in range(2):
        L.rpx_reduce_sum_f64(dx.ptr, n, res.ptr, red.ptr, rb, None, None)
        assert res.to_array()[0] == x.sum()
        L.rpx_scan_exclusive_f64(dx.ptr, y.ptr, n, scr.ptr, sb, None, None)
        assert np.array_equal(y.to_array(), np.r_[0, np.cumsum(x)[:-1]])
