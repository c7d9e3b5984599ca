"""JACOBI_2D's default plan at sizes whose fastest tile is the narrow one of
sixteen wavefronts with five rows each, against the two-sweep oracle, bit for
bit."""

import pytest

from test_gpu_jacobi_blocks import run

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,tsteps", [(1113, 117), (1131, 11), (1162, 10), (1193, 11)])
def test_tall_tiles(rpx, orc, rng, N, tsteps):
    run(rpx, orc, rng, N, tsteps)
