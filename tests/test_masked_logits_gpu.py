"""Logits-fed losses leave masked rows unread."""

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("vocab", [5, 257, 4096])  # all scalar, ragged rows (every alignment), full vectors
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_masked_rows_are_zero_and_change_nothing(vocab, dtype):
    from rl_kernel_amd.ops.logp import differentiable_logp_pair_fp32

    dev, n = torch.device("cuda"), 37
    g = torch.Generator().manual_seed(vocab)
    policy = torch.randn(n, vocab, generator=g).to(dtype).to(dev)
    ref = torch.randn(n, vocab, generator=g).to(dtype).to(dev)
    ids = torch.randint(0, vocab, (n,), generator=g).to(dev)
    mask = (torch.rand(n, generator=g) < 0.6).to(dev)
    up = torch.randn(n, generator=g).to(dev) * mask
    out = []
    for rows in (None, mask):
        x = policy.clone()
        junk = ids.clone()
        if rows is not None:  # what stands at masked positions does not matter
            x[~mask] = float("nan")
            junk[~mask] = -100
        x.requires_grad_(True)
        lp, lr = differentiable_logp_pair_fp32(x, ref, junk, rows)
        lp.backward(up)
        out.append((lp.detach(), lr, x.grad))
    (a, ar, ag), (b, br, bg) = out
    assert torch.equal(a[mask], b[mask]) and torch.equal(ar[mask], br[mask])
    assert torch.all(b[~mask] == 0) and torch.all(br[~mask] == 0)
    assert torch.equal(ag, bg) and torch.all(bg[~mask] == 0)
