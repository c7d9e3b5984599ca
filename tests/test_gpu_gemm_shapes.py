"""FP64 GEMM at sizes that reach every workgroup tile, with ragged edges and K
remainders, against 80-bit sums of sampled entries within the forward-error
bound 2(nk+2) eps |alpha| (|A||B|)ij + 2 eps |beta C0|; nothing outside C is
written."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

EPS = np.finfo(np.float64).eps


@pytest.mark.parametrize("beta", [False, True])
@pytest.mark.parametrize("ni,nj,nk", [(15, 17, 129), (63, 65, 1027), (300, 301, 7), (511, 509, 333), (700, 901, 65),
                                      (1001, 999, 100), (2047, 2049, 33), (2500, 3001, 31), (3, 4099, 17),
                                      (4099, 1, 40)])
def test_gemm_f64_shapes(rpx, rng, ni, nj, nk, beta):
    A, B, C0 = rng.uniform(-1, 1, (ni, nk)), rng.uniform(-1, 1, (nk, nj)), rng.uniform(-1, 1, ni * nj + 2)
    dA, dB = rpx.DeviceBuffer.from_array(A.reshape(-1)), rpx.DeviceBuffer.from_array(B.reshape(-1))
    dC = rpx.DeviceBuffer.from_array(C0)
    tune = rpx.tuning(flags=rpx.RPX_TUNE_GEMM_BETA) if beta else None
    rpx.lib().rpx_gemm_f64(dC.ptr + 8, dA.ptr, dB.ptr, 1.5, 1.2, ni, nj, nk, tune, None)
    out = dC.to_array()
    assert out[0] == C0[0] and out[-1] == C0[-1]
    got, old = out[1:-1].reshape(ni, nj), C0[1:-1].reshape(ni, nj)
    assert np.all(np.isfinite(got))
    i, j = np.r_[0, ni - 1, rng.integers(0, ni, 400)], np.r_[0, nj - 1, rng.integers(0, nj, 400)]
    a, b = A[i].astype(np.longdouble), B[:, j].T.astype(np.longdouble)
    ref = 1.5 * (a * b).sum(1) + (np.longdouble(1.2) * old[i, j] if beta else 0)
    bound = 2 * (nk + 2) * EPS * 1.5 * (np.abs(a) * np.abs(b)).sum(1) + 2 * EPS * 1.2 * np.abs(old[i, j])
    assert np.all(np.abs(got[i, j] - ref) <= bound)
