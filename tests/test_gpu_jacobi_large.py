"""JACOBI_2D of few time steps on large grids, where the default plan goes from
tiles to streaming chunks, against the two in-place sweeps, bit for bit."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,tsteps", [(7672, 5), (7680, 5), (8824, 5), (8832, 5), (9848, 2), (9856, 2), (9856, 3), (9856, 4), (9860, 4),
                                      (15872, 6)])
def test_few_steps_on_a_large_grid(rpx, N, tsteps):
    L, grids = rpx.lib(), []
    for fused in (True, False):
        A, B = rpx.DeviceBuffer(8 * N * N), rpx.DeviceBuffer(8 * N * N)
        L.rpx_fill_uniform_f64(A.ptr, N * N, 11, 1, -1.0, 1.0, None)
        L.rpx_fill_uniform_f64(B.ptr, N * N, 11, 2, -1.0, 1.0, None)
        if fused:
            sb = L.rpx_jacobi2d_fused_scratch_bytes(N)
            scratch = rpx.DeviceBuffer(sb)
            L.rpx_jacobi2d_fused_f64(A.ptr, B.ptr, N, tsteps, scratch.ptr, sb, None, None)
        else:
            L.rpx_jacobi2d_f64(A.ptr, B.ptr, N, tsteps, None, None)
        grids.append((A.to_array(), B.to_array()))
    for got, want in zip(*grids):
        assert np.array_equal(got, want)
