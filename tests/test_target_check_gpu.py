"""Range check of token ids in front of the launches that use them."""

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 1023, 1024, 1025, 9000])  # edges of the one workgroup's walk
def test_target_check_finds_the_one_bad_id(n):
    from rl_kernel_amd import _native

    dev = torch.device("cuda")
    ids = torch.randint(0, 50, (n,), device=dev)
    assert not _native.TargetCheck(ids, 50).out_of_range()
    for value in (-1, 50, -100):
        bad = ids.clone()
        bad[n - 1] = value
        assert _native.TargetCheck(bad, 50).out_of_range()
        mask = torch.ones(n, dtype=torch.bool, device=dev)
        assert _native.TargetCheck(bad, 50, mask=mask).out_of_range()
        mask[n - 1] = False
        assert not _native.TargetCheck(bad, 50, mask=mask).out_of_range()
    assert not _native.TargetCheck(bad, 50, ignore_index=-100).out_of_range()
    assert not _native.TargetCheck(ids[:0], 50).out_of_range()


def test_a_bad_target_raises_and_the_next_call_is_clean():
    from rl_kernel_amd.ops.linear_logp import RocmFusedLinearLogpOp

    dev, op = torch.device("cuda"), RocmFusedLinearLogpOp()
    hidden = torch.randn(300, 256, device=dev).to(torch.bfloat16).requires_grad_(True)
    weight = torch.randn(1000, 256, device=dev).to(torch.bfloat16)
    ids = torch.randint(0, 1000, (300,), device=dev)
    bad = ids.clone()
    bad[299] = 1000
    with torch.cuda.stream(torch.cuda.Stream()):  # the check belongs to the caller's stream
        torch.cuda.current_stream().wait_stream(torch.cuda.default_stream())
        with pytest.raises(ValueError, match=r"expected \[0, 999\], got \[\d+, 1000\]"):
            op(hidden, weight, bad)
        out = op(hidden, weight, ids)
        out.sum().backward()
    torch.cuda.synchronize()
    assert torch.isfinite(out).all() and torch.isfinite(hidden.grad).all()


@pytest.mark.parametrize("n", [1, 1023, 1025, 9000])
def test_marked_ids_are_a_copy_with_the_masked_ones_out_of_range(n):
    from rl_kernel_amd import _native

    dev = torch.device("cuda")
    ids = torch.randint(0, 50, (n,), device=dev)
    mask = torch.rand(n, device=dev) < 0.6
    for m in (mask, None):
        marked = torch.full_like(ids, 77)
        assert not _native.TargetCheck(ids, 50, mask=m, marked=marked).out_of_range()
        assert torch.equal(marked, ids if m is None else torch.where(m, ids, torch.full_like(ids, -1)))
