"""What becomes of the logits that a training forward keeps: hooks that hand saved tensors back elsewhere, further
backwards, several forwards before one backward, captured passes."""

import gc

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


# padded, moved and split tiles of the 16-bit kernels, chunks of the fp32 ones
@pytest.mark.parametrize("n,h,v,dtype", [
    (1, 256, 256, torch.bfloat16),
    (17, 320, 257, torch.bfloat16),
    (100, 448, 2300, torch.float16),
    (128, 512, 1300, torch.bfloat16),
    (129, 576, 1300, torch.float16),
    (192, 768, 1300, torch.bfloat16),
    (193, 832, 1300, torch.bfloat16),
    (255, 1024, 511, torch.bfloat16),
    (256, 1024, 512, torch.float16),
    (300, 1088, 1281, torch.bfloat16),
    (1000, 1024, 9000, torch.bfloat16),
    (64, 512, 33000, torch.bfloat16),
    (1, 128, 3, torch.float32),
    (63, 130, 1001, torch.float32),
    (513, 256, 1026, torch.float32),
    (2900, 128, 50001, torch.float32),
])
def test_logits_computed_again_give_the_bits_of_kept_ones(n, h, v, dtype):
    from rl_kernel_amd.ops import linear_logp as LL

    hidden, weight, bias, ids, grad = (t.detach() for t in inputs(dtype, n, h, v))
    keys = dict(temperature=0.8, ignore_index=-100)
    _, lse, _, kept = LL.fused_linear_logp_forward(hidden, weight, ids, bias, keep=True, **keys)
    want = LL.fused_linear_logp_backward(grad, hidden, weight, ids, lse, bias, kept=kept, **keys)
    got = LL.fused_linear_logp_backward(grad, hidden, weight, ids, lse, bias, as_kept=True, **keys)
    for a, b in zip(got, want):
        assert torch.equal(a, b)
    dh, _, db = LL.fused_linear_logp_backward(grad, hidden, weight, ids, lse, bias, as_kept=True, need_weight=False,
                                              **keys)
    assert torch.equal(dh, want[0]) and torch.equal(db, want[2])


def test_the_ctypes_route_and_the_compiled_one_are_the_same_calls(monkeypatch):
    from rl_kernel_amd import _compiled
    from rl_kernel_amd.ops import linear_logp as LL

    hidden, weight, bias, ids, grad = (t.detach() for t in inputs(n=150))

    def passes():
        _, lse, _, kept = LL.fused_linear_logp_forward(hidden, weight, ids, bias, keep=True, ignore_index=-100)
        return [g for as_kept in (False, True) for typed in (False, True)
                for g in LL.fused_linear_logp_backward(
                    grad, hidden, weight, ids, lse, bias, ignore_index=-100, typed_weight=typed, as_kept=as_kept,
                    kept=None if as_kept else kept.clone())]

    want = passes()
    monkeypatch.setattr(_compiled, "module", lambda: None)
    assert all(torch.equal(a, b) for a, b in zip(passes(), want))


@pytest.mark.parametrize("norm", [False, True])
@pytest.mark.parametrize("dtype,h", [(torch.bfloat16, 1024), (torch.float32, 256)])
def test_a_backward_that_was_left_no_logits_does_not_make_them(dtype, h, norm):
    """Behind saved-tensor hooks and in a second backward the fp32 logits are not stored again: beyond the
    gradients there is the workspace, with dZ in the 16-bit type where the inputs have one."""
    import ctypes

    from rl_kernel_amd import _native
    from rl_kernel_amd.ops import linear_logp as LL

    hidden, weight, _, ids, grad = inputs(dtype, 1000, h, 9000)
    keys = dict(ignore_index=-100)
    if norm:
        keys["norm_weight"] = torch.ones(h, device="cuda", dtype=dtype)
    op, need = get_op(), ctypes.c_size_t(0)
    query = _native.load().rlk_linear_logp_rmsnorm_bwd_as_kept_workspace_bytes if norm else \
        _native.load().rlk_linear_logp_bwd_as_kept_workspace_bytes
    assert query(1000, h, 9000, LL._DTYPES[dtype], ctypes.byref(need)) == 0

    def backward(logp, **more):
        base = torch.cuda.memory_allocated()
        torch.cuda.reset_peak_memory_stats()
        grads = torch.autograd.grad(logp, [hidden, weight], grad, **more)
        extra = torch.cuda.max_memory_allocated() - base - sum(g.nbytes for g in grads)
        return grads, extra

    plain = op(hidden, weight, ids, **keys)
    first, with_kept = backward(plain, retain_graph=True)
    second, extra = backward(plain)
    assert extra <= need.value + (1 << 20)
    # the logits themselves are no part of `with_kept`: dZ adds no more than it needs
    dz = 1024 * 36 * 256 * 2 if dtype == torch.bfloat16 else LL._kept_bytes(hidden, weight)
    assert extra <= with_kept + dz + (1 << 20)
    with torch.autograd.graph.saved_tensors_hooks(lambda t: t, lambda t: t):
        logp = op(hidden, weight, ids, **keys)
    third, extra = backward(logp)
    assert extra <= need.value + (1 << 20)
    for a, b, c in zip(first, second, third):
        assert torch.equal(a, b) and torch.equal(a, c)


def grpo_inputs(n):
    g = torch.Generator(device="cuda").manual_seed(3)
    rand = lambda: torch.randn(1, n, device="cuda", generator=g)
    return (torch.ones(1, n, device="cuda", dtype=torch.bool), rand() - 11, rand() - 11,
            torch.randn(1, device="cuda", generator=g))


@pytest.mark.parametrize("form", ["plain", "norm", "grpo"])
def test_many_forwards_before_one_backward_share_one_bound(form):
    """Six micro-batches whose losses are summed would hold six buffers of 206 MB; together they stay within the
    bound, the rest is computed again, and every gradient is the one it is alone."""
    from rl_kernel_amd.ops import linear_logp as LL
    from rl_kernel_amd.registry import kernel_registry

    n, h, v, calls = 1024, 1024, 50257, 6
    hidden, weight, _, ids, grad = inputs(torch.bfloat16, n, h, v)
    ids = ids.clamp_min(0)
    op, step = get_op(), kernel_registry.get_op("grpo_step_from_hidden") if form == "grpo" else None
    norm = dict(norm_weight=torch.ones(h, device="cuda", dtype=torch.bfloat16)) if form == "norm" else {}
    rest = grpo_inputs(n)

    def call(x):
        if form == "grpo":
            return step(x[None], weight, ids[None], *rest)[0]
        return (op(x, weight, ids, **norm) * grad).sum()

    xs = [(hidden.detach() * (1 + k / 8)).requires_grad_(True) for k in range(calls)]
    alone = [torch.autograd.grad(call(x), [x, weight]) for x in xs[-2:]]
    size = LL._kept_bytes(hidden, weight)
    assert calls * size > LL._KEPT_BOUND > 3 * size
    base = torch.cuda.memory_allocated()
    losses = [call(x) for x in xs]
    held = torch.cuda.memory_allocated() - base
    assert 3 * size < held < LL._KEPT_BOUND + calls * (64 * n + 4096)  # beside the logits O(n) a call
    got = torch.autograd.grad(sum(losses), xs)
    for a, b in zip(alone, got[-2:]):
        assert torch.equal(a[0], b)
    del losses, got
    assert not LL._KeptShare._alive
    # a call whose backward never comes gives its share back when it dies, and so does one that raises
    call(xs[0])
    with pytest.raises(ValueError):
        op(hidden, weight, ids + v)
    gc.collect()  # the traceback's frames
    assert not LL._KeptShare._alive


@pytest.mark.parametrize("n,slabs", [(1, 2), (64, 2), (65, 2), (128, 2), (129, 3), (192, 3), (193, 4), (255, 4)])
def test_few_tokens_hold_only_the_slabs_they_fill(n, slabs):
    hidden, weight, bias, ids, grad = inputs(torch.bfloat16, n, 1024, 5000)
    op = get_op()
    op(hidden, weight, ids, bias, ignore_index=-100)
    base = torch.cuda.memory_allocated()
    logp = op(hidden, weight, ids, bias, ignore_index=-100)
    held = torch.cuda.memory_allocated() - base
    assert 20 * slabs * (64 << 10) <= held < 20 * slabs * (64 << 10) + (32 << 10)
    torch.autograd.grad(logp, [hidden, weight, bias], grad)


@pytest.mark.parametrize("norm", [False, True])
def test_a_call_can_be_told_to_keep_none(norm):
    hidden, weight, _, ids, grad = inputs()
    keys = dict(ignore_index=-100)
    if norm:
        keys["norm_weight"] = torch.ones(H, device="cuda", dtype=torch.bfloat16)
    op = get_op()
    want = torch.autograd.grad(op(hidden, weight, ids, **keys), [hidden, weight], grad)
    for limit in (0, KEPT - 1, KEPT):
        base = torch.cuda.memory_allocated()
        logp = op(hidden, weight, ids, kept_logits_bytes=limit, **keys)
        assert (torch.cuda.memory_allocated() - base >= KEPT) == (limit == KEPT)
        got = torch.autograd.grad(logp, [hidden, weight], grad)
        assert torch.equal(got[0], want[0]) and torch.equal(got[1], want[1])
    with pytest.raises(ValueError):
        op(hidden, weight, ids, kept_logits_bytes=-1, **keys)


def test_behind_the_norm_the_workspace_counts():
    """8192 rows of 12288 beside 839 MB of logits: more than the bound on the two together, so none are kept."""
    dev = torch.device("cuda")
    x = torch.randn(8192, 12288, device=dev, dtype=torch.bfloat16).requires_grad_(True)
    weight = (torch.randn(25600, 12288, device=dev) * 0.01).to(torch.bfloat16).requires_grad_(True)
    ids = torch.randint(0, 25600, (8192,), device=dev)
    gain = torch.ones(12288, device=dev, dtype=torch.bfloat16)
    torch.cuda.synchronize()
    base = torch.cuda.memory_allocated()
    logp = get_op()(x, weight, ids, norm_weight=gain)
    assert torch.cuda.memory_allocated() - base < 100 << 20
    assert all(torch.isfinite(g).all() for g in torch.autograd.grad(logp.sum(), [x, weight]))


@pytest.mark.parametrize("dtype,h,as_kept", [(torch.bfloat16, 1024, False), (torch.bfloat16, 1024, True),
                                             (torch.float32, 250, False), (torch.float32, 250, True)])
def test_a_captured_pass_replays_with_kept_logits(dtype, h, as_kept):
    """Forward and backward in one HIP graph: every replay fills the logits again before the backward uses them
    up, and equals the eager pass on the same inputs."""
    from rl_kernel_amd.ops import linear_logp as LL

    n, v = 700, 3000
    hidden, weight, bias, ids, grad = (t.detach() for t in inputs(dtype, n, h, v))
    keys = dict(temperature=0.9, ignore_index=-100)

    def step():
        logp, lse, _, *kept = LL.fused_linear_logp_forward(hidden, weight, ids, bias, keep=not as_kept,
                                                           strict_targets=None, **keys)
        return logp, *LL.fused_linear_logp_backward(grad, hidden, weight, ids, lse, bias, as_kept=as_kept,
                                                    kept=None if as_kept else kept[0], **keys)

    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        step()
    torch.cuda.current_stream().wait_stream(side)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=side):
        out = step()
    for k in range(3):
        hidden.copy_(torch.randn(n, h, device="cuda").to(dtype))
        grad.copy_(torch.randn(n, device="cuda"))
        graph.replay()
        torch.cuda.synchronize()
        got = [t.clone() for t in out]
        assert torch.isfinite(torch.randn(1 << 20, device="cuda").sum())  # eager work and a synchronisation between
        for a, b in zip(got, step()):
            assert torch.equal(a, b), f"replay {k} differs"
