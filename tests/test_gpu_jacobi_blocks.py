"""JACOBI_2D's default plan (register-resident tiles) against the two-sweep
oracle, bit for bit: grids around one tile, odd and even, launch counts of
both parities, boundaries of A and B that differ."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def run(rpx, orc, rng, N, tsteps, scratch=True):
    A0, B0 = rng.standard_normal(N * N), rng.standard_normal(N * N)
    dA, dB = rpx.DeviceBuffer.from_array(A0), rpx.DeviceBuffer.from_array(B0)
    sb = rpx.lib().rpx_jacobi2d_fused_scratch_bytes(N) if scratch else 0
    Q = rpx.DeviceBuffer.from_array(np.full(N * N, np.nan)) if scratch else None
    rpx.lib().rpx_jacobi2d_fused_f64(dA.ptr, dB.ptr, N, tsteps, Q.ptr if Q else None, sb, None, None)
    A, B = orc.jacobi2d(A0, B0, N, tsteps)
    assert np.array_equal(dA.to_array(), A)
    assert np.array_equal(dB.to_array(), B)


@pytest.mark.parametrize("N", [3, 4, 5, 33, 63, 64, 65, 127, 128])
@pytest.mark.parametrize("tsteps", [1, 2, 37])
def test_one_tile(rpx, orc, rng, N, tsteps):
    run(rpx, orc, rng, N, tsteps)


@pytest.mark.parametrize("N", [129, 130, 131, 200, 229, 256, 515, 1002, 2049])
@pytest.mark.parametrize("tsteps", [2, 3, 4, 15, 29, 44])
def test_tiles(rpx, orc, rng, N, tsteps):
    run(rpx, orc, rng, N, tsteps)


@pytest.mark.parametrize("N", [65, 131])
def test_odd_grid_without_scratch(rpx, orc, rng, N):
    run(rpx, orc, rng, N, 5, scratch=False)
