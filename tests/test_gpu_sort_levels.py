"""SORT across its two levels of splitters and into its overfull buckets: the
longest segment cut once and the shortest cut twice, segments of both kinds
beside uncut ones in one call, and buckets that a planted sample overfills, as
a replay of the sampling on the host confirms."""

import numpy as np
import pytest

from test_gpu_sort_paths import check, images, keys

pytestmark = pytest.mark.gpu

AIM, CAP = 4096, 7664      # least mean of keys per bucket; keys that one workgroup sorts at once
ONE_LEVEL = 512 * AIM      # longest segment cut by one level of splitters


@pytest.mark.parametrize("kind", ["uniform", "equal", "mostly_equal", "integers", "sorted", "bits"])
@pytest.mark.parametrize("n", [ONE_LEVEL, ONE_LEVEL + 1])
def test_longest_cut_once_and_shortest_cut_twice(rpx, kind, n):
    check(rpx, keys(kind, n, np.random.default_rng(n)), [0, n])


@pytest.mark.parametrize("kind", ["uniform", "mostly_equal", "bits"])
def test_two_levels_beside_shorter_segments(rpx, kind):
    lens = [3, 0, 4097, 1, 5000, ONE_LEVEL + 77, 0, CAP, CAP + 1, 70_000, 2 * ONE_LEVEL + 5, 1000, 0, ONE_LEVEL, 2]
    offs = [int(v) for v in np.r_[7, 7 + np.cumsum(lens)]]
    check(rpx, keys(kind, offs[-1] + 9, np.random.default_rng(6)), offs)


def test_two_levels_of_equal_segments(rpx):
    n = ONE_LEVEL + 3
    check(rpx, keys("uniform", 3 * n, np.random.default_rng(8)), [0, n, 2 * n, 3 * n])


def test_two_levels_beside_many_short_segments(rpx):
    lens = [10] * 20_000 + [ONE_LEVEL + 5] + [9] * 20_000
    check(rpx, keys("uniform", sum(lens), np.random.default_rng(9)), [int(v) for v in np.r_[0, np.cumsum(lens)]])


def mix64(z):
    z = (z ^ (z >> np.uint64(30))) * np.uint64(0xBF58476D1CE4E5B9)
    z = (z ^ (z >> np.uint64(27))) * np.uint64(0x94D049BB133111EB)
    return z ^ (z >> np.uint64(31))


def cut(n):
    """Buckets of a segment of n keys cut once, and how many keys are sampled for them."""
    samples = lambda k: 2048 if k <= 16 else 8192
    k = -(-n // AIM)
    for _ in range(3):
        spread = np.sqrt(np.float32(k) / np.float32(samples(k)))
        aim = int(np.float32(CAP) / (np.float32(1) + np.float32(4.5) * spread))
        if aim > AIM:
            k = -(-n // aim)
    k = max(k, 2)
    return k, samples(k)


def sampled_places(n, samples):
    with np.errstate(over="ignore"):
        i = np.arange(samples, dtype=np.uint64)
        jitter = mix64(i * np.uint64(0x9E3779B97F4A7C15) + np.uint64(n)) >> np.uint64(48)
        place = (i << np.uint64(16) | jitter) * np.uint64(n)
    return (place >> np.uint64(16 + samples.bit_length() - 1)).astype(np.int64)


# Pieces of the overfull bucket, for 1, 2, 2, 3, 3 and 5 rounds of merging.
@pytest.mark.parametrize("n,pieces", [(9000, 2), (17_000, 3), (30_000, 4), (32_500, 5), (40_000, 5), (150_000, 19)])
@pytest.mark.parametrize("kind", ["uniform", "bits"])
def test_overfull_bucket(rpx, n, pieces, kind):
    """Every sampled key above every other one: the first bucket gets all the rest
    and its share of the sample."""
    rng = np.random.default_rng(n)
    k, samples = cut(n)
    places = sampled_places(n, samples)
    x = keys(kind, n, rng)
    x[np.isnan(x) & (images(x) >> np.uint64(63) == 1)] = 0.5  # nothing above the planted keys
    x = np.where(x > 1e300, 1.0, x)
    x[places] = rng.uniform(1.1e300, 1.2e300, samples)
    splitters = np.sort(x[places])[[j * samples // k for j in range(1, k)]]
    first = np.count_nonzero(images(x) < images(splitters[:1]))
    assert -(-first // CAP) == pieces, (k, first)
    check(rpx, x, [0, n])
