"""SCAN of long arrays on the scratch of an earlier segmented SCAN whose
offsets lie where the long array's look-back words go, exact on integers."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("start", [21_000_000, 37_748_736 + 5])  # epochs 1 and 2 of the words, were they bare
def test_long_scan_after_far_segments(rpx, rng, start):
    L = rpx.lib()
    n = 5_000_011
    x = rng.integers(-9, 10, n).astype(float)
    far = rng.integers(-9, 10, 10).astype(float)
    dx, y = rpx.DeviceBuffer.from_array(x), rpx.DeviceBuffer(8 * n)
    big, out = rpx.DeviceBuffer(8 * (start + 10)), rpx.DeviceBuffer(8 * (start + 10))
    L.rpx_memcpy_h2d(big.ptr + 8 * start, far.ctypes.data, 80)
    # One segment: its table is the 64-bit words 96..99 behind the header, the place of tiles 96..99 of 306.
    o = rpx.offsets_array([start, start + 10])
    sb = max(L.rpx_scan_scratch_bytes(n, None), L.rpx_scan_segmented_scratch_bytes(o, 1))
    scr = rpx.DeviceBuffer(sb)
    L.rpx_scan_scratch_init(scr.ptr, sb, None)
    for _ in range(4):
        L.rpx_scan_exclusive_segmented_f64(big.ptr, out.ptr, o, 1, scr.ptr, sb, None)
        L.rpx_scan_exclusive_f64(dx.ptr, y.ptr, n, scr.ptr, sb, None, None)
        assert np.array_equal(y.to_array(), np.r_[0, np.cumsum(x)[:-1]])
        got = np.empty(10)
        L.rpx_memcpy_d2h(got.ctypes.data, out.ptr + 8 * start, 80)
        assert np.array_equal(got, np.r_[0, np.cumsum(far)[:-1]])
    assert L.rpx_scan_scratch_status(scr.ptr) == 0
