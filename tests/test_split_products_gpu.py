"""The fp32 kernels multiply fp32 operands as sums of three bf16 pieces: as accurate against float64 as
fp32 arithmetic is, over the whole exponent range, and exact about infinities and NaN."""

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
