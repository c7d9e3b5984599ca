"""SORT of keys that its double network orders only after a shift of their
images, or not at all: NaNs of one sign and of both, infinities, and spans at
the limit of the shift and one above it, in buckets and in samples."""

import numpy as np
import pytest

from test_gpu_sort_paths import check

pytestmark = pytest.mark.gpu

NAN, MINUS_NAN, LEAST_NAN, INF, MINUS_INF = 0x7FF8 << 48, 0xFFF8 << 48, (0x7FF0 << 48) + 1, 0x7FF0 << 48, 0xFFF0 << 48
LARGEST, MINUS_LARGEST = (0x7FF0 << 48) - 1, (0xFFF0 << 48) - 1
PLANTED = {  # bit patterns strewn among normal keys
    "nan": [NAN], "minus_nan": [MINUS_NAN], "nan_payloads": [LEAST_NAN, NAN, NAN + 5, (1 << 63) - 1],
    "minus_inf": [MINUS_INF], "zeros_and_nan": [NAN, 0, 1 << 63, 1, (1 << 63) + 1],
    "widest_that_fits": [MINUS_INF, LARGEST], "one_too_wide": [MINUS_LARGEST, LEAST_NAN],
    "infinities": [MINUS_INF, INF], "both_nans": [NAN, MINUS_NAN], "all": [(1 << 63) - 1, (1 << 64) - 1],
}


@pytest.mark.parametrize("planted", PLANTED)
@pytest.mark.parametrize("n", [2, 900, 2048, 3000, 7664, 8000, 100_000])
def test_special_keys(rpx, planted, n):
    rng = np.random.default_rng(n)
    x = rng.normal(size=n)
    at = rng.integers(0, n, max(len(PLANTED[planted]), n // 50))
    x.view(np.uint64)[at] = np.resize(np.array(PLANTED[planted], dtype=np.uint64), len(at))
    check(rpx, x, [0, n])


@pytest.mark.parametrize("bits", [NAN, MINUS_NAN, MINUS_INF, INF])
def test_only_special_keys(rpx, bits):
    x = np.full(20_000, np.array([bits], dtype=np.uint64).view(np.float64)[0])
    check(rpx, x, [0, 100, 20_000])
