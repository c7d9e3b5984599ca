"""GPU: mixed-precision GEMM where its moduli go to one workgroup each, to a few
or to all, rows longer than a work-item keeps, and column exponents in one part
or in the most, against the stated bound on a long double product."""

import numpy as np
import pytest

from test_gpu_gemm_mixed import exact, run_mixed, stated_bound

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ni,nj,nk,moduli", [
    (1, 1, 1, 0), (1, 1, 1, 1), (256, 256, 255, 16), (255, 257, 1025, 0),  # a workgroup per modulus
    (1300, 2100, 40, 0), (1100, 1600, 130, 7),  # groups of several, the last one smaller
    (40, 30, 4095, 0), (40, 30, 4097, 0), (9, 70, 8193, 0), (3, 2, 40_000, 0), (3, 2, 131_071, 3)])
def test_mixed_gemm_groups(rpx, ni, nj, nk, moduli):
    rng = np.random.default_rng(ni + nk)
    A = rng.uniform(-1, 1, ni * nk) * np.exp2(rng.integers(-3, 4, ni * nk))
    B = rng.uniform(-1, 1, nk * nj) * np.exp2(rng.integers(-3, 4, nk * nj))
    if nk > 1000:  # the largest of a column in its last part
        B.reshape(nk, nj)[-1] *= 64.0
    C = run_mixed(rpx, A, B, -0.75, ni, nj, nk, moduli)
    bound, _ = stated_bound(rpx, A, B, -0.75, ni, nj, nk, moduli)
    assert np.all(np.abs(C - exact(A, B, -0.75, ni, nj, nk)) <= bound)
