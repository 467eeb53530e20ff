"""Token counts and vocabularies that no 256-wide tile divides: the last token tile and the last vocab
tile of the 16-bit kernels are moved back to end at the edge, fewer tokens than a tile are padded."""

import pytest
import torch

from oracle import oracle as O

pytestmark = pytest.mark.gpu

# fp32 sums of exact 16-bit products: about 1e-6 on log-probs of magnitude 10
LOGP_ATOL = 2e-5
# one rounding of dZ to the input type (2^-9 bf16, 2^-12 f16 at most, random signs) and one of the result
GRAD_REL = {torch.bfloat16: 5e-3, torch.float16: 1e-3}


@pytest.fixture(scope="module")
def dev():
    return torch.device("cuda")


def make(n, h, v, dtype, bias, seed):
    g = torch.Generator().manual_seed(seed)
    hidden = torch.randn(n, h, generator=g).to(dtype)
    weight = (torch.randn(v, h, generator=g) * 0.05).to(dtype)
    b = torch.randn(v, generator=g) * 0.3 if bias else None
    ids = torch.randint(0, v, (n,), generator=g)
    ids[:min(n, 3)] = torch.tensor([v - 1, max(0, v // 256 * 256 - 1), 0])[:min(n, 3)]
    if n > 8:
        ids[n // 2] = -100
    return hidden, weight, b, ids, torch.randn(n, generator=g)


def rel(a, b):
    return ((a.float().cpu() - b).norm() / b.norm().clamp_min(1e-30)).item()


# token counts around the 64-row K steps and the 256-row tiles; vocabularies likewise, the smallest
# that the moved tile takes among them; several chunks and pieces (small budgets) with short last ones
@pytest.mark.parametrize("n,h,v,dtype,bias,budget", [
    (1, 256, 256, torch.bfloat16, False, 0),
    (16, 256, 257, torch.bfloat16, True, 0),
    (63, 320, 319, torch.float16, False, 0),
    (64, 256, 1000, torch.bfloat16, False, 0),
    (65, 256, 8200, torch.bfloat16, True, 0),
    (160, 512, 9000, torch.float16, False, 0),
    (255, 256, 511, torch.bfloat16, False, 0),
    (257, 256, 577, torch.bfloat16, True, 0),
    (300, 384, 50257 // 4, torch.bfloat16, False, 0),
    (511, 576, 769, torch.float16, True, 0),
    (513, 256, 1281, torch.bfloat16, True, 256 << 10),
    (1000, 256, 2100, torch.bfloat16, False, 1 << 20),
    (1025, 1024, 33000, torch.bfloat16, True, 0),
])
def test_ragged_edges_match_the_oracle(dev, n, h, v, dtype, bias, budget):
    from rl_kernel_amd.ops import linear_logp as LL

    hidden, weight, b, ids, grad = make(n, h, v, dtype, bias, 7 * n + v)
    keys = dict(temperature=0.8, ignore_index=-100)
    ref = O.linear_logp(hidden, weight, ids, b, **keys)
    r_dh, r_dw, r_db = O.linear_logp_backward(grad, hidden, weight, ids, b, **keys)
    hd, wd, td, gd = hidden.to(dev), weight.to(dev), ids.to(dev), grad.to(dev)
    bd = b.to(dev) if bias else None
    logp, lse, err = LL.fused_linear_logp_forward(hd, wd, td, bd, **keys)
    assert int(err) == 0
    assert (logp.cpu() - ref).abs().max().item() < LOGP_ATOL
    runs = [LL.fused_linear_logp_backward(gd, hd, wd, td, lse, bd, dz_budget_bytes=budget, typed_weight=t, **keys)
            for t in (False, False, True)]
    dh, dw, db = runs[0]
    assert rel(dh, r_dh) < GRAD_REL[dtype] and rel(dw, r_dw) < GRAD_REL[dtype]
    if bias:
        assert rel(db, r_db) < GRAD_REL[dtype]
    assert torch.equal(dh, runs[1][0]) and torch.equal(dw, runs[1][1])
    # the typed weight gradient is the fp32 sum rounded once
    assert runs[2][1].dtype == dtype and torch.equal(runs[2][1], dw.to(dtype))
    assert torch.equal(dh, runs[2][0])
    assert torch.all(dh.float().cpu()[ids == -100] == 0)
    # rows are independent of the batch: every row of its own tile against the whole call
    alone, _, _ = LL.fused_linear_logp_forward(hd[-1:].contiguous(), wd, td[-1:].contiguous(), bd, **keys)
    assert abs(float(alone[0]) - float(logp[-1])) < LOGP_ATOL


@pytest.mark.parametrize("n", [100, 8192 + 77])
def test_typed_weight_gradient_behind_the_norm(dev, n):
    from rl_kernel_amd.ops import linear_logp as LL

    hidden, weight, _, ids, grad = make(n, 256, 1100, torch.bfloat16, False, n)
    gain = (1.0 + 0.1 * torch.randn(256, generator=torch.Generator().manual_seed(1))).to(dev)
    hd, wd, td, gd = hidden.to(dev), weight.to(dev), ids.to(dev), grad.to(dev)
    _, lse, _ = LL.fused_norm_linear_logp_forward(hd, gain, wd, td, ignore_index=-100)
    a = LL.fused_norm_linear_logp_backward(gd, hd, gain, wd, td, lse, ignore_index=-100)
    b = LL.fused_norm_linear_logp_backward(gd, hd, gain, wd, td, lse, ignore_index=-100, typed_weight=True)
    assert torch.equal(a[0], b[0]) and torch.equal(a[1], b[1])
    assert b[2].dtype == torch.bfloat16 and torch.equal(b[2], a[2].to(torch.bfloat16))


def test_target_rows_next_to_the_moved_tile(dev):
    """Targets in the rows that the moved last tile shares with its neighbour are picked up once."""
    from rl_kernel_amd.ops import linear_logp as LL

    n, h, v = 300, 256, 700  # last tile: rows 444 .. 699, its own from 512 on
    hidden, weight, _, _, _ = make(n, h, v, torch.bfloat16, False, 3)
    ids = torch.arange(400, 700)
    ref = O.linear_logp(hidden, weight, ids)
    logp, _, _ = LL.fused_linear_logp_forward(hidden.to(dev), weight.to(dev), ids.to(dev))
    assert (logp.cpu() - ref).abs().max().item() < LOGP_ATOL
