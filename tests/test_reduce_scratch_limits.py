"""DOT and REDUCE_SUM refuse a scratch below the two-level layout of their
length, also where the slots of a short reduction would fit in it."""

import pytest

from rajaperf_amd import abi


@pytest.mark.parametrize("n", [1, 10, 4097, 20_000])
def test_small_scratch_is_refused(n):
    L = abi.lib()
    align = lambda b: -(-b // 256) * 256
    tickets = 256 + 256 + 256 + align(8 * -(-n // (512 * 32)))  # header, one group's ticket and sum, partials
    slots = 256 + 16 * -(-n // 4096)
    assert slots < tickets <= L.rpx_reduce_scratch_bytes(n, None)
    for size in (0, 255, slots, tickets - 1):  # nothing is launched: the pointers are never read
        assert L.raw("rpx_dot_f64")(4096, 8192, n, 16384, 0, 32768, size, None, None) == abi.RPX_ERR_SCRATCH_TOO_SMALL
        assert L.raw("rpx_reduce_sum_f64")(4096, n, 16384, 32768, size, None, None) == abi.RPX_ERR_SCRATCH_TOO_SMALL
