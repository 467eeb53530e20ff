"""Heads whose logits share a large negative offset: every log-sum-exp lies far below zero, so a row that
does not exist (padding up to a tile, a neighbour's row) must not meet a real row's log-sum-exp."""

import pytest
import torch

from oracle import oracle as O

pytestmark = pytest.mark.gpu

OFFSET = -200.0
# The offset is the last column, so a running fp32 sum reaches 200 with its last products: one rounding to
# ulp(200) = 2^-16 there, one of the bias, for the target and for the log-sum-exp each
LOGP_ATOL = 4 * 2.0 ** -16
# one rounding of dZ to the input type (2^-9 bf16, 2^-12 f16 at most, random signs) and one of the result
GRAD_REL = {torch.bfloat16: 5e-3, torch.float16: 1e-3}


def make(n, h, v, dtype, bias, seed):
    g = torch.Generator().manual_seed(seed)
    hidden = torch.randn(n, h, generator=g)
    weight = torch.randn(v, h, generator=g) * 0.05
    hidden[:, -1], weight[:, -1] = 4.0, OFFSET / 4.0
    # a bias that takes back half of the offset: the bias alone is 100 above every log-sum-exp
    b = torch.randn(v, generator=g) * 0.3 - OFFSET / 2 if bias else None
    ids = torch.randint(0, v, (n,), generator=g)
    if n > 8:
        ids[n // 2] = -100
    return hidden.to(dtype), weight.to(dtype), b, ids, torch.randn(n, generator=g)


def rel(a, b):
    return ((a.float().cpu() - b).norm() / b.norm().clamp_min(1e-30)).item()


# fewer tokens than a tile (padded), 128 (whole K steps), a moved last token tile, a hidden size that the
# chained kernels do not take
@pytest.mark.parametrize("n,h", [(1, 256), (100, 256), (128, 320), (255, 256), (300, 256), (100, 72)])
@pytest.mark.parametrize("dtype,bias", [(torch.bfloat16, False), (torch.bfloat16, True), (torch.float16, True)])
def test_gradients_stay_finite_and_match_the_oracle(n, h, dtype, bias):
    from rl_kernel_amd.ops import linear_logp as LL

    dev, v = torch.device("cuda"), 577
    hidden, weight, b, ids, grad = make(n, h, v, dtype, bias, n + h)
    z = hidden.double() @ weight.double().t() + (b.double() if bias else 0.0)
    ref = z.gather(1, ids.clamp_min(0)[:, None])[:, 0] - torch.logsumexp(z, 1)
    ref[ids == -100] = 0.0
    r_dh, r_dw, r_db = O.linear_logp_backward(grad, hidden, weight, ids, b, ignore_index=-100)
    hd, wd, td, gd = hidden.to(dev), weight.to(dev), ids.to(dev), grad.to(dev)
    bd = b.to(dev) if bias else None
    logp, lse, _ = LL.fused_linear_logp_forward(hd, wd, td, bd, ignore_index=-100)
    assert lse.max().item() < -80
    assert (logp.double().cpu() - ref).abs().max().item() < LOGP_ATOL
    for typed in (False, True):
        dh, dw, db = LL.fused_linear_logp_backward(gd, hd, wd, td, lse, bd, typed_weight=typed, ignore_index=-100)
        assert torch.isfinite(dw).all() and (db is None or torch.isfinite(db).all())
        # (the last column of dH is the offset times a sum that cancels: nothing but rounding)
        assert rel(dh[:, :-1], r_dh[:, :-1]) < GRAD_REL[dtype] and rel(dw, r_dw) < GRAD_REL[dtype]
        if bias:
            assert rel(db, r_db) < GRAD_REL[dtype]


@pytest.mark.parametrize("n", [77, 8192 + 77])  # the only block, and a short last one behind a full block
def test_short_last_block_behind_the_norm(n):
    from rl_kernel_amd.ops import linear_logp as LL

    dev, h, v = torch.device("cuda"), 256, 577
    g = torch.Generator().manual_seed(n)
    x = torch.randn(n, h, generator=g).to(torch.bfloat16)
    weight = torch.randn(v, h, generator=g) * 0.05
    x[:, 0], weight[:, 0] = 1.0, -2.0
    weight = weight.to(torch.bfloat16)
    gain = torch.ones(h)
    gain[0] = 100.0  # the offset: column 0 of the normalised rows is about 100
    b = torch.randn(v, generator=g) * 0.3
    ids, grad = torch.randint(0, v, (n,), generator=g), torch.randn(n, generator=g)
    rows = O.rms_norm(x, gain, eps=1e-6)
    _, r_dw, r_db = O.linear_logp_backward(grad, rows, weight, ids, b)
    xd, gd, wd, td, bd = x.to(dev), gain.to(dev), weight.to(dev), ids.to(dev), b.to(dev)
    _, lse, _ = LL.fused_norm_linear_logp_forward(xd, gd, wd, td, bd)
    assert lse.max().item() < -80
    d_x, d_gain, d_w, d_b = LL.fused_norm_linear_logp_backward(grad.to(dev), xd, gd, wd, td, lse, bd)
    for t in (d_x, d_gain, d_w, d_b):
        assert torch.isfinite(t).all()
    # (column 0 is a hundred times the others)
    assert rel(d_w[:, 1:], r_dw[:, 1:]) < GRAD_REL[torch.bfloat16] and rel(d_b, r_db) < GRAD_REL[torch.bfloat16]


@pytest.mark.parametrize("n", [1, 100, 255, 300])
def test_a_logit_of_minus_infinity_gets_no_gradient(n):
    """A weight row that is -inf in a column where every hidden value is positive: its logits are -inf, its
    probability and its gradient 0, and no other row's gradient meets an infinity or NaN."""
    from rl_kernel_amd.ops import linear_logp as LL

    dev, h, v = torch.device("cuda"), 256, 577
    hidden, weight, b, ids, grad = make(n, h, v, torch.bfloat16, True, n)
    hidden[:, 3] = hidden[:, 3].abs() + 0.5
    weight[7, 3] = weight[576, 3] = float("-inf")
    ids = ids.clamp(8, 575)
    hd, wd, td, bd = hidden.to(dev), weight.to(dev), ids.to(dev), b.to(dev)
    _, lse, _ = LL.fused_linear_logp_forward(hd, wd, td, bd)
    assert torch.isfinite(lse).all()
    _, dw, db = LL.fused_linear_logp_backward(grad.to(dev), hd, wd, td, lse, bd, need_hidden=False)
    assert torch.isfinite(dw).all() and torch.isfinite(db).all()
    assert torch.all(dw[[7, 576]] == 0) and torch.all(db[[7, 576]] == 0)
