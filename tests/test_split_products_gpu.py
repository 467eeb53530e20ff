"""The fp32 kernels multiply fp32 operands as sums of three bf16 pieces: as accurate against float64 as
fp32 arithmetic is, whatever the length and sign of the sums, down to where fp32 itself loses bits, and
exact about infinities and NaN."""

import pytest
import torch

pytestmark = pytest.mark.gpu

# fp32 products and running fp32 sums of K terms of random sign: about sqrt(K) * 2^-24 of a term's size
# per result, the same share of the result's norm; twice that for the two contractions of a gradient
EPS = 2.0 ** -24


@pytest.fixture(scope="module")
def dev():
    return torch.device("cuda")


def exact(hidden, weight, ids, grad):
    h, w = hidden.double(), weight.double()
    z = h @ w.t()
    lse = torch.logsumexp(z, 1)
    logp = z.gather(1, ids[:, None])[:, 0] - lse
    dz = torch.softmax(z, 1) * -grad.double()[:, None]
    dz.scatter_add_(1, ids[:, None], grad.double()[:, None])
    return logp, dz @ w, dz.t() @ h


# one K step, ragged K (element-wise loads), K steps around the three LDS stages, several tiles
@pytest.mark.parametrize("n,h,v", [(40, 16, 300), (70, 33, 257), (300, 48, 513), (513, 1024, 3000), (256, 2048, 40)])
@pytest.mark.parametrize("spread", [0, 20])
def test_error_against_float64_is_that_of_fp32(dev, n, h, v, spread):
    from rl_kernel_amd.ops import linear_logp as LL

    g = torch.Generator().manual_seed(n + v + spread)
    hidden = torch.randn(n, h, generator=g)
    weight = torch.randn(v, h, generator=g) * h ** -0.5
    if spread:  # exponents far apart inside a row, products of ordinary size
        e = torch.randint(-spread, spread + 1, (h,), generator=g).float()
        hidden, weight = hidden * 2.0 ** e, weight * 2.0 ** -e
    ids = torch.randint(0, v, (n,), generator=g)
    grad = torch.randn(n, generator=g)
    want = exact(hidden, weight, ids, grad)
    hd, wd, td = hidden.to(dev), weight.to(dev), ids.to(dev)
    logp, lse, _ = LL.fused_linear_logp_forward(hd, wd, td)
    dh, dw, _ = LL.fused_linear_logp_backward(grad.to(dev), hd, wd, td, lse)
    # a column of dH / dW has the scale of its exponent: compare column by column
    col = lambda a, b: ((a.double().cpu() - b).norm(dim=0) / b.norm(dim=0).clamp_min(1e-300)).max().item()
    assert (logp.double().cpu() - want[0]).abs().max().item() < 8 * EPS * (h ** 0.5 + 12)
    assert col(dh, want[1]) < 2 * EPS * (max(h, v, n) ** 0.5 + 16)
    assert col(dw, want[2]) < 2 * EPS * (max(h, v, n) ** 0.5 + 16)


def test_infinities_and_nan_stay_what_they_are(dev):
    """A weight row that is -inf in a column where every hidden value is positive has logit -inf, leaves
    the softmax and takes nobody with it; a NaN row of hidden states stays alone."""
    from rl_kernel_amd.ops import linear_logp as LL

    n, h, v = 70, 40, 600
    g = torch.Generator().manual_seed(5)
    hidden, weight = torch.randn(n, h, generator=g), torch.randn(v, h, generator=g) * 0.2
    hidden[:, 3] = hidden[:, 3].abs() + 0.1
    weight[7, 3] = weight[300, 3] = float("-inf")
    ids = torch.randint(8, 299, (n,), generator=g)
    ids[0] = 7
    hidden[5, 11] = float("nan")
    want = torch.log_softmax(hidden.double() @ weight.double().t(), 1).gather(1, ids[:, None])[:, 0]
    logp, _, _ = LL.fused_linear_logp_forward(hidden.to(dev), weight.to(dev), ids.to(dev))
    logp = logp.double().cpu()
    assert logp[0] == float("-inf") and torch.isnan(logp[5]) and torch.isnan(want[5])
    rest = torch.tensor([i for i in range(n) if i not in (0, 5)])
    assert (logp[rest] - want[rest]).abs().max().item() < 1e-5


# one and several stages of 16, a ragged one, sums long enough for a bias to show
@pytest.mark.parametrize("k", [8, 16, 40, 256, 1024, 4096, 16384])
@pytest.mark.parametrize("one_sign", [False, True])
def test_error_of_a_dot_product_is_that_of_rounding_to_nearest(dev, k, one_sign):
    """A head of one row: lse is the logit itself, up to two roundings.  A stage of 16 products is rounded
    into the running sum once, by at most 2^-24 of it and 0.58 * 2^-24 rms: over K / 16 stages of one
    sign, which grow linearly, 0.58 * sqrt(K / 16 / 3), of random sign less.  The stage's own roundings, lse's
    two and what the pieces leave out: 1.5."""
    from rl_kernel_amd.ops import linear_logp as LL

    g = torch.Generator().manual_seed(k)
    draw = torch.rand if one_sign else torch.randn
    hidden, weight = draw(2048, k, generator=g), draw(1, k, generator=g)
    z = (hidden.double() @ weight.double().t())[:, 0]
    size = (hidden.double().abs() @ weight.double().abs().t())[:, 0]
    _, lse, _ = LL.fused_linear_logp_forward(hidden.to(dev), weight.to(dev), torch.zeros(2048, dtype=torch.long).to(dev))
    err = (lse.double().cpu() - z) / size / EPS
    assert err.square().mean().sqrt().item() < 1.5 + 0.58 * (k / 48) ** 0.5


# operands around 2^-115 and 2^-120, whose lower pieces bf16 cannot hold: hidden states (K-contiguous in the
# logits, K-major in dW), the weight (K-contiguous, K-major in dH) and dZ through the upstream gradient
@pytest.mark.parametrize("hidden_exp,weight_exp,grad_exp", [(-120, 120, 0), (120, -120, 0), (0, 0, -115)])
@pytest.mark.parametrize("h", [64, 61])  # whole stages of aligned groups, element-wise loads
def test_tiny_operands_keep_their_bits(dev, h, hidden_exp, weight_exp, grad_exp):
    from rl_kernel_amd.ops import linear_logp as LL

    n, v = 256, 1000
    g = torch.Generator().manual_seed(h - hidden_exp)
    hidden = torch.randn(n, h, generator=g) * 2.0 ** hidden_exp
    weight = torch.randn(v, h, generator=g) * h ** -0.5 * 2.0 ** weight_exp
    ids, grad = torch.randint(0, v, (n,), generator=g), torch.randn(n, generator=g) * 2.0 ** grad_exp
    want = exact(hidden, weight, ids, grad)
    hd, wd, td = hidden.to(dev), weight.to(dev), ids.to(dev)
    logp, lse, _ = LL.fused_linear_logp_forward(hd, wd, td)
    dh, dw, _ = LL.fused_linear_logp_backward(grad.to(dev), hd, wd, td, lse)
    assert (logp.double().cpu() - want[0]).abs().max().item() < 8 * EPS * (h ** 0.5 + 12)
    for got, ref in ((dh, want[1]), (dw, want[2])):
        rel = ((got.double().cpu() - ref).norm() / ref.norm()).item()
        assert rel < 2 * EPS * (v ** 0.5 + 16)


def test_a_logit_beyond_the_largest_float_is_an_infinity(dev):
    """hi * hi passes -3.4e38, lo * hi the other way: the logit is -inf as in fp32, and nobody else's."""
    from rl_kernel_amd.ops import linear_logp as LL

    n, h, v = 70, 40, 600
    g = torch.Generator().manual_seed(6)
    hidden, weight = torch.randn(n, h, generator=g), torch.randn(v, h, generator=g) * 0.2
    hidden[:, 3], weight[:, 3] = 3e6 * (1.0 + torch.rand(n, generator=g)), 0.0
    weight[7, 3] = -3.3e38
    weight[300:310, 3] = -3.2e38 * (1.0 + 0.05 * torch.rand(10, generator=g))
    ids = torch.randint(8, 299, (n,), generator=g)
    ids[0] = 7
    logp, _, _ = LL.fused_linear_logp_forward(hidden.to(dev), weight.to(dev), ids.to(dev))
    keep = torch.tensor([i for i in range(v) if i != 7 and not 300 <= i < 310])
    z = hidden.double() @ weight.double().t()
    want = z.gather(1, ids[:, None])[:, 0] - torch.logsumexp(z[:, keep], 1)
    logp = logp.double().cpu()
    assert logp[0] == float("-inf")
    assert (logp[1:] - want[1:]).abs().max().item() < 1e-5
