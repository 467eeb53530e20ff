"""Host rules of the kept logits: what a training step holds beyond its inputs and outputs stays below 1 GB."""

import ctypes
import random
import threading

import torch


def test_kept_logits_and_workspace_stay_below_one_gigabyte():
    from rl_kernel_amd import _native

    lib, rng, kept_some = _native.load(), random.Random(3), 0
    for _ in range(3000):
        n = int(2 ** rng.uniform(0, 18))
        h = rng.choice((256, 512, 896, 1024, 1536, 2048, 4096, 4160, 8192))
        v = int(2 ** rng.uniform(8, 18))
        dtype = rng.choice((0, 1, 2))
        kept, ws = ctypes.c_size_t(0), ctypes.c_size_t(0)
        assert lib.rlk_linear_logp_kept_bytes(n, h, v, dtype, ctypes.byref(kept)) == 0
        rc = lib.rlk_linear_logp_bwd_kept_workspace_bytes(n, h, v, dtype, ctypes.byref(ws))
        if kept.value == 0:
            assert rc == -2
            continue
        kept_some += 1
        tiles = -(-n // 256) * -(-v // 256)
        assert rc == 0 and kept.value == (n * -(-v // 4) * 16 if dtype == 2 else tiles * (256 << 10)) <= 800 << 20
        assert kept.value + ws.value <= 10 ** 9, (n, h, v)
    assert kept_some > 500


def test_behind_the_norm_kept_logits_and_workspace_stay_below_one_gigabyte():
    from rl_kernel_amd import _native

    lib, rng, kept_some, refused = _native.load(), random.Random(4), 0, 0
    sizes = [(8192, 8192, 25600, 0), (8192, 12288, 25600, 0), (8192, 16384, 25600, 0), (8193, 1024, 25600, 0)]
    for _ in range(3000):
        sizes.append((int(2 ** rng.uniform(0, 14)), rng.choice((896, 1024, 2048, 4096, 8192, 12288, 16384)),
                      int(2 ** rng.uniform(8, 18)), rng.choice((0, 1, 2))))
    for n, h, v, dtype in sizes:
        kept, head, ws, again = (ctypes.c_size_t(0) for _ in range(4))
        assert lib.rlk_linear_logp_rmsnorm_kept_bytes(n, h, v, dtype, ctypes.byref(kept)) == 0
        assert lib.rlk_linear_logp_kept_bytes(n, h, v, dtype, ctypes.byref(head)) == 0
        if n > 8192 or head.value == 0:
            assert kept.value == 0
            continue
        assert lib.rlk_linear_logp_rmsnorm_bwd_kept_workspace_bytes(n, h, v, dtype, ctypes.byref(ws)) == 0
        assert lib.rlk_linear_logp_rmsnorm_bwd_as_kept_workspace_bytes(n, h, v, dtype, ctypes.byref(again)) == 0
        fits = head.value + ws.value <= 10 ** 9
        assert kept.value == (head.value if fits else 0), (n, h, v)
        # fp32 chunks are whole 256-row tiles
        dz = -(-n // 256) * 256 * -(-v // 4) * 16 if dtype == 2 else head.value // 2
        assert again.value <= dz + ws.value + 256, (n, h, v, dtype)
        kept_some += fits
        refused += not fits
    assert kept_some > 500 and refused >= 3


def test_sizes_that_keep_none():
    from rl_kernel_amd import _native

    lib, kept = _native.load(), ctypes.c_size_t(1)
    for n, h, v, dtype in ((32768, 4096, 128256, 0), (100, 64, 5000, 2), (32768, 2048, 32000, 2), (100, 1000, 5000, 0), (100, 192, 5000, 0),
                           (100, 1024, 255, 0), (1000, 704, 5000, 0), (1638 * 2, 4096, 128256, 1)):
        assert lib.rlk_linear_logp_kept_bytes(n, h, v, dtype, ctypes.byref(kept)) == 0 and kept.value == 0
    assert lib.rlk_linear_logp_kept_bytes(0, 1024, 5000, 0, ctypes.byref(kept)) == -1


def test_a_torch_that_does_not_tell_its_hooks_keeps_none(monkeypatch):
    from rl_kernel_amd.ops import linear_logp as LL

    assert LL._may_keep()
    with torch.autograd.graph.saved_tensors_hooks(lambda t: t, lambda t: t):
        assert not LL._may_keep()
    monkeypatch.delattr(torch._C._autograd, "_top_saved_tensors_default_hooks")
    assert not LL._may_keep()


def test_shares_of_all_threads_stay_within_the_bound():
    from rl_kernel_amd.ops.linear_logp import _KEPT_BOUND, _KeptShare

    here, there = torch.device("cuda", 0), torch.device("cuda", 1)
    size, held, most = _KEPT_BOUND // 5 - 1, [], []

    def work(seed):
        rng, mine = random.Random(seed), []
        for _ in range(400):
            if mine and rng.random() < 0.5:
                mine.pop()
            else:
                share = _KeptShare.take(here, size)
                if share is not None:
                    mine.append(share)
            most.append(sum(b for _, b in list(_KeptShare._alive.values())))
        held.append(mine)

    threads = [threading.Thread(target=work, args=(k,)) for k in range(8)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert max(most) == 5 * size <= _KEPT_BOUND
    others = [_KeptShare.take(there, size) for _ in range(6)]  # another device has its own
    assert others[4] is not None and others[5] is None
    held.clear()
    others.clear()
    del t, threads
    assert not _KeptShare._alive and _KeptShare.take(here, _KEPT_BOUND) and _KeptShare.take(here, _KEPT_BOUND + 1) is None


def test_a_buffer_holds_the_slabs_that_have_tokens():
    from rl_kernel_amd import _native

    lib, kept, least = _native.load(), ctypes.c_size_t(0), ctypes.c_size_t(0)
    for n, quarters in ((1, 2), (64, 2), (128, 2), (129, 3), (192, 3), (193, 4), (255, 4), (256, 4), (1000, 4)):
        for dtype in (0, 1, 2):
            assert lib.rlk_linear_logp_kept_bytes(n, 4096, 50257, dtype, ctypes.byref(kept)) == 0
            assert lib.rlk_linear_logp_kept_least_bytes(n, 4096, 50257, dtype, ctypes.byref(least)) == 0
            assert least.value == (kept.value if dtype == 2 else kept.value * quarters // 4) > 0
        # one byte less is refused before anything is launched (no pointer is followed)
        assert lib.rlk_linear_logp_fwd_kept(16, 16, None, 16, 16, 16, 256, 1 << 40, n, 4096, 50257, 0, 1, 1.0, 0, 0, 0,
                                            None, 16, kept.value * quarters // 4 - 1, None) == -1
        assert b"buffer too small" in lib.rlk_last_error()
    assert lib.rlk_linear_logp_kept_least_bytes(100, 64, 5000, 0, ctypes.byref(least)) == 0 and least.value == 0
