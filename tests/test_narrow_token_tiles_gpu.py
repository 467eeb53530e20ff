"""Forwards of at most 192 tokens run on a narrower token tile; a token's bits are those of the full tile."""

import pytest
import torch

pytestmark = pytest.mark.gpu


# the edges of the tiles of 64, 128 and 192 tokens
@pytest.mark.parametrize("n", [1, 63, 64, 65, 128, 129, 191, 192, 193])
@pytest.mark.parametrize("h,v,dtype", [(192, 1000, torch.bfloat16), (512, 20000, torch.float16)])
def test_few_tokens_have_the_bits_of_a_full_tile(n, h, v, dtype):
    from rl_kernel_amd.ops import linear_logp as LL

    dev = torch.device("cuda")
    g = torch.Generator().manual_seed(v)
    hidden = torch.randn(256, h, generator=g).to(dtype).to(dev)
    weight, ref = ((torch.randn(v, h, generator=g) * 0.05).to(dtype).to(dev) for _ in range(2))
    bias = (torch.randn(v, generator=g) * 0.3).to(dev)
    ids = torch.randint(0, v, (256,), generator=g).to(dev)
    keys = dict(temperature=0.7)
    full = LL.fused_linear_logp_forward(hidden, weight, ids, bias, **keys)
    exact = torch.log_softmax((hidden.double() @ weight.double().T + bias.double()) / 0.7, 1)
    assert (full[0].double() - exact.gather(1, ids[:, None])[:, 0]).abs().max().item() < 2e-5
    few = LL.fused_linear_logp_forward(hidden[:n].contiguous(), weight, ids[:n].contiguous(), bias, **keys)
    assert torch.equal(few[0], full[0][:n]) and torch.equal(few[1], full[1][:n])
    pair = LL.fused_linear_logp_forward_pair(hidden[:n].contiguous(), weight, ref, ids[:n].contiguous(), **keys)
    alone = LL.fused_linear_logp_forward(hidden, ref, ids, **keys)
    assert torch.equal(pair[2], alone[0][:n]) and torch.equal(pair[3], alone[1][:n])
