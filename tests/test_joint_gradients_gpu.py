"""dH and dW of one dZ block share a launch: which workgroup takes a tile, and what it did before, must
not show in the tile's bits."""

import pytest
import torch

from oracle import oracle as O

pytestmark = pytest.mark.gpu

# one rounding of dZ to the input type (2^-9, random signs) and one of the result
GRAD_REL = 5e-3


# dH items (token tiles x h tiles x parts) and dW tiles (vocab tiles x h tiles) against the 256 workgroups: fewer
# than a launch of 256; a last round of dH items with few and with most workgroups in it; whole rounds of
# either; split dH tiles; several chunks and pieces with short last ones
@pytest.mark.parametrize("n,h,v,budget", [
    (100, 256, 300, 0),              # 1 + 2 items
    (2304, 8192, 513, 0),            # 288 + 96: 32 workgroups with a second dH tile
    (3900, 4096, 1000, 0),           # 256 + 64: whole rounds
    (3000, 4160, 2300, 0),           # 204 + 153: the last h tile is moved back
    (700, 1024, 20000, 0),           # 12 tiles in 19 parts + 316
    (1500, 512, 9000, 1 << 20),      # many blocks, the last chunk and piece short
])
def test_joint_launch_equals_the_gradients_alone(n, h, v, budget):
    from rl_kernel_amd.ops import linear_logp as LL

    dev = torch.device("cuda")
    g = torch.Generator().manual_seed(n + v)
    hidden = torch.randn(n, h, generator=g).to(torch.bfloat16)
    weight = (torch.randn(v, h, generator=g) * 0.03).to(torch.bfloat16)
    ids = torch.randint(0, v, (n,), generator=g)
    up = torch.randn(n, generator=g)
    hd, wd, td, ud = hidden.to(dev), weight.to(dev), ids.to(dev), up.to(dev)
    _, lse, _ = LL.fused_linear_logp_forward(hd, wd, td)
    keys = dict(dz_budget_bytes=budget)
    both = LL.fused_linear_logp_backward(ud, hd, wd, td, lse, **keys)
    only_h = LL.fused_linear_logp_backward(ud, hd, wd, td, lse, need_weight=False, **keys)
    only_w = LL.fused_linear_logp_backward(ud, hd, wd, td, lse, need_hidden=False, **keys)
    assert torch.equal(both[0], only_h[0]) and only_h[1] is None
    assert torch.equal(both[1], only_w[1]) and only_w[0] is None
    r_dh, r_dw, _ = O.linear_logp_backward(up, hidden, weight, ids)
    for out, ref in ((both[0], r_dh), (both[1], r_dw)):
        assert ((out.float().cpu() - ref).norm() / ref.norm()).item() < GRAD_REL
