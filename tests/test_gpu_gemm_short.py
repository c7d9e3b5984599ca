"""FP64 GEMM of short K at sizes that reach its 64 x 128 tiles, inside C and on
its ragged edges, with K remainders, within the bound of the other shapes'
test."""

import pytest

import test_gpu_gemm_shapes as shapes

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("beta", [False, True])
@pytest.mark.parametrize("ni,nj,nk", [(1024, 2048, 16), (1087, 2111, 17), (64, 32_768, 9), (2048, 2049, 1),
                                      (2047, 2048, 64), (3000, 2500, 33), (1281, 4097, 130), (4096, 4096, 200),
                                      (4096, 4096, 300)])
def test_gemm_short_k(rpx, rng, ni, nj, nk, beta):
    shapes.test_gemm_f64_shapes(rpx, rng, ni, nj, nk, beta)
