"""What becomes of the logits that a training forward keeps: hooks that hand saved tensors back elsewhere, further
backwards, several forwards before one backward, captured passes."""

import pytest
import torch

pytestmark = pytest.mark.gpu

N, H, V = 300, 1024, 5000
KEPT = 2 * 20 * (256 << 10)  # whole 256 x 256 tiles of fp32


def inputs(dtype=torch.bfloat16, n=N, h=H, v=V):
    dev = torch.device("cuda")
    g = torch.Generator().manual_seed(n + v)
    hidden = torch.randn(n, h, generator=g).to(dtype).to(dev).requires_grad_(True)
    weight = (torch.randn(v, h, generator=g) * 0.03).to(dtype).to(dev).requires_grad_(True)
    bias = (torch.randn(v, generator=g) * 0.3).to(dev).requires_grad_(True)
    ids = torch.randint(0, v, (n,), generator=g)
    ids[n // 2] = -100
    return hidden, weight, bias, ids.to(dev), torch.randn(n, generator=g).to(dev)


def get_op():
    from rl_kernel_amd.registry import kernel_registry

    return kernel_registry.get_op("linear_logp")


def shifted_copy(t):
    """The same values one element off every 16-byte boundary."""
    flat = torch.empty(t.numel() + 1, device=t.device, dtype=t.dtype)
    return flat[1:].copy_(t.detach().reshape(-1)).view(t.shape)


@pytest.mark.parametrize("norm", [False, True])
@pytest.mark.parametrize("dtype,tol", [(torch.bfloat16, 5e-3), (torch.float32, 1e-5)])
def test_unpacked_tensors_may_lie_off_the_16_byte_boundary(dtype, tol, norm):
    """Tolerance: one rounding of dZ and one of the result to the input type; fp32 sums in another order."""
    hidden, weight, _, ids, grad = inputs(dtype)
    keys = dict(ignore_index=-100)
    if norm:
        keys["norm_weight"] = torch.ones(H, device="cuda", dtype=dtype)
    op = get_op()
    plain = torch.autograd.grad(op(hidden, weight, ids, **keys), [hidden, weight], grad)
    unpack = lambda t: shifted_copy(t) if t.is_floating_point() and t.dim() == 2 else t
    with torch.autograd.graph.saved_tensors_hooks(lambda t: t, unpack):
        logp = op(hidden, weight, ids, **keys)
    for got, want in zip(torch.autograd.grad(logp, [hidden, weight], grad), plain):
        assert ((got.float() - want.float()).norm() / want.float().norm()).item() < tol
