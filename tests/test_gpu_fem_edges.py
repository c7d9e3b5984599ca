"""MASS3DPA and DIFFUSION3DPA bit-exact against the oracle where the last
workgroup is full, one element short or holds one element (floor(256/Q1D^2)
elements each)."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("d1d", range(2, 9))
@pytest.mark.parametrize("short", [-1, 0, 1])
def test_fem_workgroup_edges(rpx, orc, rng, d1d, short):
    q1d = d1d + 1
    NE = 2 * (256 // q1d ** 2) + short
    b, g = rng.uniform(-1, 1, q1d * d1d), rng.uniform(-1, 1, q1d * d1d)
    X, Y0 = rng.uniform(-1, 1, NE * d1d ** 3), rng.uniform(-1, 1, NE * d1d ** 3)
    for op in ("mass", "diffusion"):
        D = rng.uniform(-1, 1, NE * (1 if op == "mass" else 6) * q1d ** 3)
        bufs = [rpx.DeviceBuffer.from_array(a) for a in (b, g, D, X, np.r_[Y0, 7.5])]
        p = [x.ptr for x in bufs]
        if op == "mass":
            rpx.lib().rpx_mass3dpa_f64(*p, NE, d1d, q1d, None, None)
            ref = orc.mass3dpa(b, g, D, X, Y0, NE, d1d, q1d)
        else:
            rpx.lib().rpx_diffusion3dpa_f64(*p, NE, d1d, q1d, 1, None, None)
            ref = orc.diffusion3dpa(b, g, D, X, Y0, NE, d1d, q1d)
        assert np.array_equal(bufs[4].to_array(), np.r_[ref, 7.5])
