"""FP64 GEMM at sizes that reach its 96 x 96, 96 x 64 and deep 64 x 64 tiles,
with ragged edges and K remainders, within the bound of the other shapes' test."""

import pytest

import test_gpu_gemm_shapes as shapes

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("beta", [False, True])
@pytest.mark.parametrize("ni,nj,nk", [(1441, 1535, 33), (1499, 1501, 70), (1536, 1536, 32), (1055, 1100, 95),
                                      (1057, 1087, 31), (1152, 1088, 64), (1021, 1023, 63), (1001, 1000, 130),
                                      (1100, 1500, 1)])
def test_gemm_tiles(rpx, rng, ni, nj, nk, beta):
    shapes.test_gemm_f64_shapes(rpx, rng, ni, nj, nk, beta)
