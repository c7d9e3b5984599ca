"""JACOBI_2D's default plan on grids that take its wide tiles, against the
two-sweep oracle, bit for bit: odd and even N, even and odd numbers of
launches, few steps and the most per launch, boundaries of A and B that
differ."""

import pytest

from test_gpu_jacobi_blocks import run

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,tsteps", [(2047, 50), (2048, 40), (2500, 40), (2501, 41), (2771, 15), (3000, 30), (4097, 6)])
def test_wide_tiles(rpx, orc, rng, N, tsteps):
    run(rpx, orc, rng, N, tsteps)
