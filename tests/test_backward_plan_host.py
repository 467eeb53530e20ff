"""Which blocks the backward takes: those of the joint dH + dW price only where it promises 2.5 % over the blocks of
three separate launches (below that the clock does not show it, and every fp32 sum would be grouped another way)."""

import ctypes

import pytest


# measured against the blocks of separate launches: 1.006, 0.976 and 0.984 (kept as they were) ...
@pytest.mark.parametrize("n,h,v,plan", [
    (12000, 2048, 151936, (8192, 16384, 2, 10)),
    (17829, 5120, 32768, (6144, 16384, 3, 2)),
    (6648, 896, 32000, (6656, 16128, 1, 2)),
    # ... 1.187, 1.154 and 1.083 (taken)
    (2273, 2048, 151936, (2304, 57344, 1, 3)),
    (3044, 1536, 201088, (3072, 36864, 1, 6)),
    (16073, 3584, 201088, (8192, 16384, 2, 13)),
    # no joint launch (H % 64 != 0)
    (3000, 1000, 50257, (3072, 25344, 1, 2)),
])
def test_blocks_change_only_for_a_gain_that_shows(n, h, v, plan):
    from rl_kernel_amd import _native

    out = (ctypes.c_int64 * 5)()
    assert _native.load().rlk_linear_logp_bwd_plan(n, h, v, 0, 0, out) == 0
    assert tuple(out)[:4] == plan
