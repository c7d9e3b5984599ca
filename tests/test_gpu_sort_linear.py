"""GPU: SORT of one bucket by its linear map (lengths at the edges of the
workgroups, bins of many keys, values the map must refuse) against numpy on the
64-bit images, bit for bit."""

import numpy as np
import pytest

from test_gpu_sort_paths import check

pytestmark = pytest.mark.gpu


def values(kind, n, rng):
    if kind == "uniform":
        return rng.uniform(-1, 1, n)
    if kind == "pairs":  # every value twice or more
        return rng.integers(0, n // 2 + 1, n).astype(np.float64)
    if kind == "few":  # bins of thousands of equal keys
        return rng.choice(np.array([-3.0, 0.25, 7.0]), n)
    if kind == "clusters":  # bins of hundreds of different keys beside empty ones
        return rng.choice(np.array([0.0, 1.0, 1e6]), n) + rng.uniform(0, 1e-9, n)
    if kind == "outlier":  # all keys but one in the first bin
        x = rng.uniform(0, 1, n)
        x[n // 2] = 1e308
        return x
    if kind == "zeros":  # -0.0 before +0.0
        return rng.choice(np.array([-1.0, -0.0, 0.0, 1.0]), n)
    if kind == "denormals":
        return rng.integers(-9, 9, n) * 5e-324
    return rng.choice(np.array([-np.finfo(float).max, np.finfo(float).max, 0.0]), n)  # a spread that overflows


@pytest.mark.parametrize("kind", ["uniform", "pairs", "few", "clusters", "outlier", "zeros", "denormals", "widest"])
@pytest.mark.parametrize("n", [2, 7, 8, 9, 15, 16, 17, 24, 25, 255, 257, 3823, 3824, 3825, 7663, 7664, 7665])
def test_one_bucket(rpx, kind, n):
    check(rpx, values(kind, n, np.random.default_rng(n)), [0, n])


@pytest.mark.parametrize("kind", ["uniform", "few", "clusters", "zeros"])
def test_both_workgroup_sizes(rpx, kind):
    # Segments of up to 3824 keys go to small workgroups, those beside a longer one to large ones.
    rng = np.random.default_rng(3)
    for lens in ([1, 3824, 16, 0, 2000], [1, 3824, 16, 0, 2000, 7664, 5]):
        offs = [3] + [int(v) for v in 3 + np.cumsum(lens)]
        check(rpx, values(kind, offs[-1] + 4, rng), offs)


@pytest.mark.parametrize("nseg", [128, 129])
def test_gathered_and_own_samples(rpx, nseg):
    # Up to 128 segments' samples are gathered by a kernel of their own.
    rng = np.random.default_rng(nseg)
    offs = [0] + [int(v) for v in np.cumsum(rng.integers(7000, 9000, nseg))]
    check(rpx, values("uniform", offs[-1], rng), offs)
    check(rpx, values("uniform", nseg * 8192, rng), [8192 * i for i in range(nseg + 1)])
