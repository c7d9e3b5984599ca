"""GPU: the paths of the segmented SORT (one bucket, one and two levels of
splitters, repeated keys, keys its double network cannot order, overfull
buckets) against numpy on the 64-bit images, bit for bit."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

ONE_LEVEL = 512 * 3072  # longest segment cut by one level of splitters


def images(x):
    b = x.view(np.uint64)
    return np.where(b >> np.uint64(63), ~b, b | np.uint64(1 << 63))


def check(rpx, x, offsets):
    d = rpx.DeviceBuffer.from_array(x)
    o = rpx.offsets_array(offsets)
    nseg = len(offsets) - 1
    sb = rpx.lib().rpx_sort_segmented_scratch_bytes(o, nseg)
    s = rpx.DeviceBuffer(sb)
    rpx.lib().rpx_sort_segmented_f64(d.ptr, o, nseg, s.ptr, sb, None)
    got, want = images(d.to_array()), images(x)
    for b, e in zip(offsets[:-1], offsets[1:]):
        want[b:e] = np.sort(want[b:e])
    assert np.array_equal(got, want)


def keys(kind, n, rng):
    if kind == "uniform":
        return rng.uniform(-1, 1, n)
    if kind == "equal":
        return np.full(n, -3.5)
    if kind == "mostly_equal":
        x = np.full(n, 2.0)
        x[rng.integers(0, n, n // 50 + 1)] = rng.normal(size=n // 50 + 1)
        return x
    if kind == "integers":
        return rng.integers(-40, 40, n).astype(np.float64)
    if kind == "sorted":
        return np.arange(n, dtype=np.float64)
    if kind == "reversed":
        return -np.arange(n, dtype=np.float64)
    bits = rng.integers(0, 1 << 64, n, dtype=np.uint64)  # any pattern: NaNs, infinities, denormals, zeros
    bits[rng.integers(0, n, n // 8 + 1)] = rng.choice(
        np.array([0, 1 << 63, 1, (1 << 63) + 1, 0x7FF0 << 48, 0xFFF0 << 48, (0x7FF0 << 48) + 1, (1 << 64) - 1],
                 dtype=np.uint64), n // 8 + 1)
    return bits.view(np.float64)


@pytest.mark.parametrize("kind", ["uniform", "equal", "mostly_equal", "integers", "sorted", "reversed", "bits"])
@pytest.mark.parametrize("n", [1, 1024, 1025, 2049, 4096, 4097, 8193, 200_001, ONE_LEVEL, ONE_LEVEL + 1, 4_000_003])
def test_sort_lengths(rpx, kind, n):
    check(rpx, keys(kind, n, np.random.default_rng(n)), [0, n])


def test_sort_mixed_lengths_in_one_call(rpx):
    # One bucket, one level and two levels of splitters side by side, odd starts, empty segments.
    lens = [3, 0, 4097, 1, 5000, ONE_LEVEL + 77, 0, 4096, 70_000, 1000]
    offs = [7] + [int(v) for v in 7 + np.cumsum(lens)]
    rng = np.random.default_rng(5)
    x = np.concatenate([rng.normal(size=offs[7]), keys("bits", offs[-1] - offs[7] + 9, rng)])
    check(rpx, x, offs)


@pytest.mark.parametrize("n", [9000, 40_000, 150_000])  # overfull buckets of 1, 5 and 19 pieces of 8192 keys
def test_sort_overfull_bucket(rpx, n):
    """Every sampled key above every other one: the first bucket gets all the rest."""
    mask = (1 << 64) - 1

    def mix64(z):
        z = ((z ^ (z >> 30)) * 0xBF58476D1CE4E5B9) & mask
        z = ((z ^ (z >> 27)) * 0x94D049BB133111EB) & mask
        return z ^ (z >> 31)

    rng = np.random.default_rng(n)
    x = rng.uniform(0, 1, n)
    at = [((i << 16 | mix64((i * 0x9E3779B97F4A7C15 + n) & mask) >> 48) * n) >> 27 for i in range(2048)]
    x[at] = rng.uniform(1, 2, 2048)
    check(rpx, x, [0, n])
