"""Small vocabularies: up to 14 tiles a token block is one run of tiles whatever the token count, below 64
tiles the runs are as long for 8192 tokens as for one, so a batch and its micro-batches sum the softmax in the
same grouping and give the same bits."""

import ctypes

import pytest
import torch

VOCABS = (256, 700, 1000, 1024, 3000, 3584)


@pytest.mark.parametrize("v", VOCABS)
@pytest.mark.parametrize("h,dtype", [(64, 0), (72, 1), (256, 0), (4096, 0), (64, 2)])
def test_schedule_does_not_follow_the_token_count(v, h, dtype):
    from rl_kernel_amd import _native

    lib, seen = _native.load(), set()
    for n in (1, 128, 256, 257, 512, 768, 2048, 4096, 32768, 1 << 20):
        plan = (ctypes.c_int64 * 4)()
        assert lib.rlk_linear_logp_fwd_plan(n, h, v, dtype, plan) == 0
        seen.add((plan[1], plan[2]))
    assert len(seen) == 1, (v, h, seen)


@pytest.mark.parametrize("v", (4096, 8192, 8448, 12000, 16128))
@pytest.mark.parametrize("h,dtype", [(64, 0), (4096, 0), (64, 2)])
def test_runs_below_64_tiles_are_the_same_for_one_and_for_8192_tokens(v, h, dtype):
    from rl_kernel_amd import _native

    lib, seen = _native.load(), set()
    for n in (1, 256, 512, 768, 2048, 5000, 8192):
        plan = (ctypes.c_int64 * 4)()
        assert lib.rlk_linear_logp_fwd_plan(n, h, v, dtype, plan) == 0
        seen.add((plan[1], plan[2]))
    assert len(seen) == 1, (v, h, seen)


@pytest.mark.gpu
@pytest.mark.parametrize("h,v,dtype", [(64, 1000, torch.bfloat16), (256, 1024, torch.bfloat16),
                                       (256, 3000, torch.float16), (64, 3000, torch.float32),
                                       (256, 4096, torch.bfloat16)])
def test_micro_batches_give_the_bits_of_the_batch(h, v, dtype):
    from rl_kernel_amd.ops import linear_logp as LL

    n, g = 2560, torch.Generator().manual_seed(v)
    hidden = torch.randn(n, h, generator=g).to(dtype).cuda()
    weight = (torch.randn(v, h, generator=g) * 0.3).to(dtype).cuda()
    ids = torch.randint(0, v, (n,), generator=g).cuda()
    logp, lse, _ = LL.fused_linear_logp_forward(hidden, weight, ids)
    for lo, hi in ((0, 256), (256, 768), (768, 2560)):
        part = LL.fused_linear_logp_forward(hidden[lo:hi], weight, ids[lo:hi])
        assert torch.equal(part[0], logp[lo:hi]) and torch.equal(part[1], lse[lo:hi])
