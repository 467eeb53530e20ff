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


@pytest.mark.parametrize("vocab", [257, 4096])
@pytest.mark.parametrize("ref_dtype", [torch.bfloat16, torch.float32])  # one launch for both tensors, two scans
def test_masked_rows_get_no_gradient_whatever_comes_from_above(vocab, ref_dtype):
    from rl_kernel_amd.ops.logp import differentiable_logp_fp32, differentiable_logp_pair_fp32

    dev, n = torch.device("cuda"), 37
    g = torch.Generator().manual_seed(vocab)
    x = (torch.randn(n, vocab, generator=g) * 3 + 200).to(torch.bfloat16).to(dev)  # exp overflows without an lse
    ids = torch.randint(0, vocab, (n,), generator=g).to(dev)
    mask = (torch.rand(n, generator=g) < 0.6).to(dev)
    up = torch.randn(n, generator=g).to(dev)
    a, b = x.clone().requires_grad_(True), x.clone().requires_grad_(True)
    lp, lr = differentiable_logp_pair_fp32(a, x.to(ref_dtype), ids, mask)
    assert torch.all(lp[~mask] == 0) and torch.all(lr[~mask] == 0)
    lp.backward(up)
    differentiable_logp_fp32(b, ids).backward(up)
    assert torch.all(a.grad[~mask] == 0) and torch.equal(a.grad[mask], b.grad[mask])


def test_ids_may_be_overwritten_before_the_backward():
    """The logits-fed losses keep a copy of the ids: a trainer that refills its buffers for the next
    micro-batch gets the gradient of the ids it passed."""
    from rl_kernel_amd.registry import kernel_registry

    dev, op = torch.device("cuda"), kernel_registry.get_op("grpo_loss")
    b, t, v = 4, 8, 100
    g = torch.Generator().manual_seed(1)
    policy, old = torch.randn(b, t, v, generator=g).to(dev), torch.randn(b, t, generator=g).to(dev) - 4
    ref, rewards = policy + 0.1, torch.randn(b, generator=g).to(dev)
    ids = torch.randint(0, v, (b, t), generator=g).to(dev)
    mask = (torch.rand(b, t, generator=g) < 0.7).to(dev)
    grads = []
    for overwrite in (False, True):
        x, i, m = policy.clone().requires_grad_(True), ids.clone(), mask.clone()
        loss, _, _ = op(x, ref, i, old, rewards, m, beta=0.1, samples_per_prompt=2)
        if overwrite:
            i.fill_(0), m.fill_(True)
        loss.backward()
        grads.append(x.grad)
    assert torch.equal(grads[0], grads[1])
