"""FP64 GEMM with an infinite alpha: every product alpha*A[i][k] of the sum is
the infinity of A's sign, and nothing that pads K to whole slabs adds a NaN.
The sizes are those at which a finite alpha reaches every workgroup tile, with
a K remainder."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("beta", [False, True])
@pytest.mark.parametrize("alpha", [np.inf, -np.inf])
@pytest.mark.parametrize("ni,nj,nk", [(15, 17, 129), (63, 65, 1027), (300, 301, 7), (511, 509, 333), (700, 901, 65),
                                      (1001, 1000, 130), (1021, 1023, 63), (1441, 1535, 33), (1499, 1501, 70),
                                      (2047, 2049, 33), (2500, 3001, 31), (3000, 3100, 10)])
def test_gemm_infinite_alpha(rpx, rng, ni, nj, nk, alpha, beta):
    dA = rpx.DeviceBuffer.from_array(rng.uniform(0.5, 1, ni * nk))
    dB = rpx.DeviceBuffer.from_array(rng.uniform(0.5, 1, nk * nj))
    dC = rpx.DeviceBuffer.from_array(rng.uniform(-1, 1, ni * nj))
    tune = rpx.tuning(flags=rpx.RPX_TUNE_GEMM_BETA) if beta else None
    rpx.lib().rpx_gemm_f64(dC.ptr, dA.ptr, dB.ptr, alpha, 1.2, ni, nj, nk, tune, None)
    assert np.all(dC.to_array() == alpha)
