"""Training steps of few logits: the forward leaves its fp32 logits for the backward, which turns them into dZ
in place instead of computing them again."""

import pytest
import torch

from oracle import oracle as O

pytestmark = pytest.mark.gpu

# one rounding of dZ to the input type (2^-9 bf16, 2^-12 f16 at most, random signs) and one of the result
# (fp32: sums of at most 2050 fp32 products against another order of them)
GRAD_REL = {torch.bfloat16: 5e-3, torch.float16: 1e-3, torch.float32: 1e-5}


def make(n, h, v, dtype, bias, seed, low=0.0):
    g = torch.Generator().manual_seed(seed)
    hidden = torch.randn(n, h, generator=g).to(dtype)
    weight = (torch.randn(v, h, generator=g) * 0.03).to(dtype)
    b = torch.randn(v, generator=g) * 0.3 + low if bias else None
    ids = torch.randint(0, v, (n,), generator=g)
    ids[:min(n, 3)] = torch.tensor([v - 1, max(0, v // 256 * 256 - 1), 0])[:min(n, 3)]
    if n > 8:
        ids[n // 2] = -100
    return hidden, weight, b, ids, torch.randn(n, generator=g)


def rel(a, b):
    return ((a.float().cpu() - b).norm() / b.norm().clamp_min(1e-30)).item()


# around the 16-token columns that are stored, the 64-token slabs and the 256-row tiles; moved token, vocab and
# hidden tiles; split dH tiles; log-sum-exps below -88
@pytest.mark.parametrize("n,h,v,dtype,bias,low", [
    (1, 256, 256, torch.bfloat16, False, 0.0),
    (17, 320, 257, torch.bfloat16, True, 0.0),
    (64, 256, 1000, torch.float16, False, 0.0),
    (100, 448, 2300, torch.bfloat16, True, -200.0),
    (255, 1024, 511, torch.float16, True, 0.0),
    (256, 1024, 512, torch.bfloat16, False, 0.0),
    (300, 1088, 1281, torch.bfloat16, True, 0.0),
    (1000, 1024, 9000, torch.bfloat16, True, 0.0),
    (1, 128, 3, torch.float32, True, 0.0),
    (63, 130, 1001, torch.float32, True, -200.0),
    (300, 257, 2050, torch.float32, True, 0.0),
    (513, 256, 1024, torch.float32, False, 0.0),
])
def test_kept_logits_give_the_gradients(n, h, v, dtype, bias, low):
    from rl_kernel_amd.ops import linear_logp as LL

    dev = torch.device("cuda")
    hidden, weight, b, ids, grad = make(n, h, v, dtype, bias, 7 * n + v, low)
    keys = dict(temperature=0.8, ignore_index=-100)
    r_dh, r_dw, r_db = O.linear_logp_backward(grad, hidden, weight, ids, b, **keys)
    hd, wd, td, gd = hidden.to(dev), weight.to(dev), ids.to(dev), grad.to(dev)
    bd = b.to(dev) if bias else None
    assert LL._kept_bytes(hd, wd) == (n * -(-v // 4) * 16 if dtype == torch.float32
                                      else -(-n // 256) * -(-v // 256) * (256 << 10))
    plain = LL.fused_linear_logp_forward(hd, wd, td, bd, **keys)

    def backward(**more):
        logp, lse, _, kept = LL.fused_linear_logp_forward(hd, wd, td, bd, keep=True, **keys)
        assert torch.equal(logp, plain[0]) and torch.equal(lse, plain[1])
        return LL.fused_linear_logp_backward(gd, hd, wd, td, lse, bd, kept=kept, **keys, **more)

    dh, dw, db = backward()
    assert rel(dh, r_dh) < GRAD_REL[dtype] and rel(dw, r_dw) < GRAD_REL[dtype]
    if bias:
        assert rel(db, r_db) < GRAD_REL[dtype]
    assert torch.all(dh.float().cpu()[ids == -100] == 0)
    again = backward()
    typed = backward(typed_weight=True)
    assert torch.equal(dh, again[0]) and torch.equal(dw, again[1])
    assert torch.equal(dh, typed[0]) and torch.equal(typed[1], dw.to(dtype))
    assert torch.equal(backward(need_weight=False)[0], dh) and torch.equal(backward(need_hidden=False)[1], dw)
    # added to what the buffers hold
    out = torch.ones_like(dw)
    db_out = torch.ones_like(db) if bias else None
    backward(weight_grad_out=out, bias_grad_out=db_out, accumulate=True)
    assert torch.allclose(out, dw + 1, rtol=1e-6, atol=1e-6)
    assert not bias or torch.allclose(db_out, db + 1, rtol=1e-6, atol=1e-6)


@pytest.mark.parametrize("norm", [False, True])
def test_one_forward_serves_any_number_of_backwards(norm):
    """The kept logits are used up by the first backward; later ones, and those behind saved-tensor hooks (which
    keep none), give the same bits, and no call holds them longer than its backward."""
    from rl_kernel_amd.registry import kernel_registry

    op = kernel_registry.get_op("linear_logp")
    dev = torch.device("cuda")
    n, h, v = 300, 1024, 5000
    hidden, weight, _, ids, grad = make(n, h, v, torch.bfloat16, False, 5)
    hd, wd = hidden.to(dev).requires_grad_(True), weight.to(dev).requires_grad_(True)
    td, gd = ids.to(dev), grad.to(dev)
    keys = dict(ignore_index=-100, norm_weight=torch.ones(h, device=dev, dtype=torch.bfloat16) if norm else None)
    kept_bytes = 2 * 20 * (256 << 10)
    op(hd, wd, td, **keys)
    base = torch.cuda.memory_allocated()
    logp = op(hd, wd, td, **keys)
    assert torch.cuda.memory_allocated() - base >= kept_bytes
    first = torch.autograd.grad(logp, [hd, wd], gd, retain_graph=True)
    held = torch.cuda.memory_allocated() - base
    assert held < kept_bytes + first[0].nbytes + first[1].nbytes
    second = torch.autograd.grad(logp, [hd, wd], gd)
    del logp
    with torch.autograd.graph.saved_tensors_hooks(lambda t: t, lambda t: t):
        base = torch.cuda.memory_allocated()
        logp = op(hd, wd, td, **keys)
        assert torch.cuda.memory_allocated() - base < kept_bytes
    third = torch.autograd.grad(logp, [hd, wd], gd)
    with torch.no_grad():
        base = torch.cuda.memory_allocated()
        scored = op(hd, wd, td, **keys)
        assert torch.cuda.memory_allocated() - base < kept_bytes
    assert torch.equal(scored, logp)
    for a, b, c in zip(first, second, third):
        assert torch.equal(a, b) and torch.equal(a, c)
