"""The work that users of this package have it do, as measurable cases.

A case is a plain dict.  ``path`` says which public entry point it goes through:

* ``score``       log-probs of given tokens from hidden states, no gradient (``linear_logp``, with
                  ``reference``: policy and frozen reference head in one call)
* ``train``       ``linear_logp`` forward and backward through autograd
* ``grpo``        ``training.grpo_loss_step`` and its backward (hidden states -> loss -> gradients)
* ``logits_logp`` selected log-probs of logits that a model has already written (``logp``)
* ``logits_grpo`` the logits-fed GRPO loss and its backward (``grpo_loss``)

Head shapes are those of the benchmark, the tests and the shape sweep of the design notes.
"""

import math

import torch

IGNORE = -100
DTYPES = {"bf16": torch.bfloat16, "f16": torch.float16, "f32": torch.float32}
BYTES = {"bf16": 2, "f16": 2, "f32": 4}

HIDDEN = (896, 1536, 2048, 2560, 2880, 3584, 4096, 5120, 8192)
VOCAB = (32000, 32768, 50257, 128256, 151936, 152064, 201088)

# tokens * hidden * vocab of the largest listed case of each kind of arithmetic
MOST_16 = 32768 * 4096 * 128256
MOST_32 = 2048 * 2048 * 32768


def head(name, path, tokens, hidden, vocab, dtype="bf16", **options):
    case = {"path": path, "tokens": tokens, "hidden": hidden, "vocab": vocab, "dtype": dtype,
            "temperature": 1.0, "ignored": 0.0, "bias": False}
    case.update({"score": {"reference": False},
                 "train": {"norm": False, "main_grad": False},
                 "grpo": {"length": 512, "group": 8, "skip_masked": False}}[path])
    case.update(options)
    return dict(case, name=name) if name else case


def logits(name, path, tokens, vocab, dtype="bf16", **options):
    case = {"path": path, "tokens": tokens, "vocab": vocab, "dtype": dtype}
    if path == "logits_grpo":
        case.update({"length": 512, "group": 8})
    case.update(options)
    return dict(case, name=name) if name else case


def listed():
    return [
        # one step of the example program's toy policy: launches and host work are all there is
        head("grpo_toy", "grpo", 128, 64, 1000, bias=True, length=16, group=4),
        # log-probs of one short answer: the weight is read once, few tokens share it
        head("score_short", "score", 160, 4096, 128256),
        # rollout log-probs of policy and reference for a few answers of uneven length
        head("score_pair", "score", 3000, 2048, 151936, reference=True, temperature=0.7),
        # a small micro-batch, a tenth of it padding
        head("train_micro", "train", 1000, 1536, 151936, ignored=0.1, temperature=0.7),
        # a head with a bias and a vocabulary that no tile divides
        head("train_odd_vocab", "train", 4096, 2048, 50257, bias=True),
        # the benchmark's step
        head("train_llama", "train", 32768, 4096, 128256),
        # f16, 1 % ignored positions, the gradient added into the trainer's fp32 buffer
        head("train_f16_main_grad", "train", 12000, 2048, 151936, "f16", ignored=0.01, main_grad=True),
        # the model's last RMSNorm goes through the op too
        head("train_norm", "train", 8192, 4096, 32000, norm=True),
        # fp32 activations and head
        head("train_f32", "train", 2048, 2048, 32768, "f32"),
        # a GRPO batch whose prompt and padding positions are left out of the head
        head("grpo_masked", "grpo", 16384, 3584, 152064, skip_masked=True, group=16),
        # log-probs of a large batch of written logits: one pass over memory
        logits("logits_logp", "logits_logp", 16384, 128256),
        # loss and gradient of written policy and reference logits
        logits("logits_grpo", "logits_grpo", 4096, 32000),
    ]


def log_uniform(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    path = rng.choices(("score", "train", "grpo", "logits_logp", "logits_grpo"), (25, 45, 14, 8, 8))[0]
    if path.startswith("logits"):
        vocab = rng.choice((1000,) + VOCAB)
        dtype = rng.choices(("bf16", "f16", "f32"), (70, 15, 15))[0]
        most = 16384 * 128256 // (BYTES[dtype] // 2)
        if path == "logits_logp":
            return logits(None, path, log_uniform(rng, 8, min(16384, most // vocab)), vocab, dtype)
        length, group = log_uniform(rng, 8, 512), rng.choice((2, 4, 8))
        sequences = group * log_uniform(rng, 1, max(1, min(16, most // 8 // (group * length * vocab))))
        return logits(None, path, sequences * length, vocab, dtype, length=length, group=group)
    dtype = rng.choices(("bf16", "f16", "f32"), (70, 20, 10))[0]
    most = MOST_32 if dtype == "f32" else MOST_16
    hidden = rng.choice(HIDDEN if dtype != "f32" else HIDDEN[:3])
    vocab = rng.choice(VOCAB if dtype != "f32" else VOCAB[:3])
    options = {"temperature": rng.choice((1.0, 1.0, 0.7)), "bias": rng.random() < 0.15}
    top = min(32768, most // (hidden * vocab))
    if path == "grpo":
        length, group = log_uniform(rng, 16, min(1024, top // 4)), rng.choice((2, 4, 8, 16))
        sequences = group * log_uniform(rng, 1, max(1, min(16, top // (group * length))))
        tokens = min(sequences, max(group, top // length // group * group)) * length
        return head(None, path, tokens, hidden, vocab, dtype, length=length, group=group,
                    skip_masked=rng.random() < 0.5, **options)
    tokens = log_uniform(rng, 16, top)
    options["ignored"] = rng.choice((0.0, 0.0, 0.01, 0.1))
    if path == "score":
        options["reference"] = rng.random() < 0.3 and 2 * tokens * hidden * vocab <= most
    else:
        kind = rng.choices(("plain", "norm", "main_grad"), (60, 20, 20))[0]
        options.update(norm=kind == "norm", main_grad=kind == "main_grad")
    return head(None, path, tokens, hidden, vocab, dtype, **options)


def _selected_logps(hidden, weight, bias, ids, temperature):
    """Plain log-probs of ``ids``, a few rows at a time (the rollout's log-probs)."""
    out = []
    for lo in range(0, hidden.size(0), 1024):
        z = torch.nn.functional.linear(hidden[lo:lo + 1024], weight, bias).float() / temperature
        out.append(z.gather(1, ids[lo:lo + 1024, None])[:, 0] - torch.logsumexp(z, 1))
    return torch.cat(out)


def _completion_mask(sequences, length, gen, dev):
    """Completions of length / 4 ... length positions, the rest is padding."""
    lens = torch.randint(max(1, length // 4), length + 1, (sequences, 1), generator=gen, device=dev)
    return torch.arange(length, device=dev)[None, :] < lens


def prepare(case, seed):
    from rl_kernel_amd.registry import kernel_registry

    dev = torch.device("cuda")
    gen = torch.Generator(device=dev).manual_seed(seed)
    dt = DTYPES[case["dtype"]]
    n, v, path = case["tokens"], case["vocab"], case["path"]

    def normal(*shape, std=1.0, dtype=dt):
        return torch.randn(*shape, generator=gen, device=dev, dtype=dtype).mul_(std)

    ids = torch.randint(0, v, (n,), generator=gen, device=dev)
    rows = torch.arange(n, device=dev)
    state = {"case": case}

    if path.startswith("logits"):
        policy = normal(n, v, std=2.0)
        policy[rows, ids] += 8.0  # sampled tokens are likely ones
        if path == "logits_logp":
            return dict(state, op=kernel_registry.get_op("logp"), logits=policy, ids=ids)
        b, t = n // case["length"], case["length"]
        ref = policy + normal(n, v, std=0.05)
        mask = _completion_mask(b, t, gen, dev)
        ids = ids.view(b, t)
        logp = torch.cat([torch.log_softmax(policy[i:i + 512].float(), 1)
                          .gather(1, ids.reshape(-1, 1)[i:i + 512])[:, 0] for i in range(0, n, 512)])
        return dict(state, op=kernel_registry.get_op("grpo_loss"),
                    logits=policy.view(b, t, v).requires_grad_(True), ref=ref.view(b, t, v), ids=ids, mask=mask,
                    old=logp.view(b, t) + normal(b, t, std=0.05, dtype=torch.float32),
                    rewards=normal(b, dtype=torch.float32))

    h = case["hidden"]
    weight = normal(v, h, std=0.02)
    bias = normal(v, std=0.1) if case["bias"] else None
    # unit-variance rows that lean towards the row of the token that was sampled from them
    lean = weight[ids].float()
    hidden = normal(n, h, dtype=torch.float32) + 6.0 * lean / lean.norm(dim=1, keepdim=True)
    hidden = hidden.to(dt)
    del lean
    if case["ignored"] > 0:
        drop = torch.rand(n, generator=gen, device=dev) < case["ignored"]
        ids = torch.where(drop, torch.full_like(ids, IGNORE), ids)
    state.update(hidden=hidden, weight=weight, bias=bias, ids=ids)

    if path == "score":
        if case["reference"]:
            state["ref_weight"] = weight + normal(v, h, std=0.002)
            state["ref_bias"] = bias.clone() if bias is not None else None
        return dict(state, op=kernel_registry.get_op("linear_logp"))

    if path == "train":
        for name in ("hidden", "weight", "bias"):
            if state[name] is not None:
                state[name].requires_grad_(True)
        state.update(op=kernel_registry.get_op("linear_logp"),
                     upstream=normal(n, std=1.0 / n, dtype=torch.float32), gain=None, main_grad=None)
        if case["norm"]:
            state["gain"] = (1.0 + normal(h, std=0.1, dtype=torch.float32)).to(dt).requires_grad_(True)
        if case["main_grad"]:
            state["main_grad"] = torch.zeros(v, h, device=dev)
        return state

    b, t = n // case["length"], case["length"]
    linear = torch.nn.Linear(h, v, bias=bias is not None, device="meta")
    linear.weight = torch.nn.Parameter(weight)
    if bias is not None:
        linear.bias = torch.nn.Parameter(bias)
    logp = _selected_logps(hidden, weight, bias, ids, case["temperature"]).view(b, t)
    return dict(state, head=linear, hidden=hidden.view(b, t, h).requires_grad_(True), ids=ids.view(b, t),
                mask=_completion_mask(b, t, gen, dev),
                old=logp + normal(b, t, std=0.05, dtype=torch.float32),
                ref=logp + normal(b, t, std=0.1, dtype=torch.float32),
                rewards=normal(b, dtype=torch.float32))


def run(state):
    case = state["case"]
    path = case["path"]
    if path == "logits_logp":
        return state["op"].apply_fp32(state["logits"], state["ids"])
    if path == "logits_grpo":
        loss, policy, kl = state["op"](state["logits"], state["ref"], state["ids"], state["old"], state["rewards"],
                                       state["mask"], beta=0.04, samples_per_prompt=case["group"])
        grad, = torch.autograd.grad(loss, [state["logits"]])
        return loss.detach(), policy.detach(), kl.detach(), grad
    if path == "score":
        keys = dict(temperature=case["temperature"], ignore_index=IGNORE)
        with torch.no_grad():
            if case["reference"]:
                return state["op"].with_reference(state["hidden"], state["weight"], state["ref_weight"], state["ids"],
                                                  state["bias"], state["ref_bias"], **keys)
            return state["op"](state["hidden"], state["weight"], state["ids"], state["bias"], **keys)
    if path == "train":
        wanted = [state["hidden"]]
        keys = dict(temperature=case["temperature"], ignore_index=IGNORE)
        if case["main_grad"]:
            keys["weight_grad_out"] = state["main_grad"]
        else:
            wanted.append(state["weight"])
        if case["norm"]:
            keys["norm_weight"] = state["gain"]
            wanted.append(state["gain"])
        if case["bias"]:
            wanted.append(state["bias"])
        logp = state["op"](state["hidden"], state["weight"], state["ids"], state["bias"], **keys)
        grads = torch.autograd.grad(logp, wanted, state["upstream"])
        return (logp.detach(), *grads, state["main_grad"])
    from rl_kernel_amd.training import grpo_loss_step

    linear = state["head"]
    step = grpo_loss_step(state["hidden"], linear, state["ids"], state["mask"], state["old"], state["ref"],
                          state["rewards"], samples_per_prompt=case["group"], beta=0.04,
                          temperature=case["temperature"], skip_masked=case["skip_masked"])
    wanted = [state["hidden"], linear.weight] + ([linear.bias] if case["bias"] else [])
    grads = torch.autograd.grad(step.loss, wanted)
    return (step.loss.detach(), step.policy_loss.detach(), step.kl.detach(), step.current_logps.detach(), *grads)


def work(case):
    """Inputs once, outputs once; the contraction once forward and twice backward, active rows only."""
    n, v, e, path = case["tokens"], case["vocab"], BYTES[case["dtype"]], case["path"]
    if path == "logits_logp":
        return {"bytes": n * v * e + n * 12, "flops": 0}
    if path == "logits_grpo":
        return {"bytes": 3 * n * v * e + n * 20, "flops": 0}
    h = case["hidden"]
    active = n * (1.0 - case["ignored"]) if path != "grpo" else n * 0.625
    once = 2.0 * active * h * v
    if path == "score":
        heads = 2 if case["reference"] else 1
        return {"bytes": n * h * e + heads * (v * h * e + n * 4) + n * 8, "flops": heads * once}
    wide = 4 * 2 * v * h if path == "train" and case["main_grad"] else v * h * e
    return {"bytes": 2 * n * h * e + v * h * e + wide + n * 16, "flops": 3 * once}


def tolerance(case):
    """Forward results are fp32 sums whatever the inputs; gradients go through one 16-bit rounding
    of the softmax term and one of the result."""
    if case["path"] in ("score", "logits_logp"):
        return {"rel": 1e-5}
    if case["dtype"] == "f32":
        # a loss is a mean of signed terms that nearly cancel
        return {"rel": 1e-4 if "grpo" in case["path"] else 1e-5}
    return {"rel": 1e-2} if case["dtype"] == "bf16" else {"rel": 2e-3}


def _exact_head(hidden, weight, bias, ids, temperature, upstream=None):
    """float64 log-probs of ``ids`` (``IGNORE`` rows: 0) and, given ``upstream(logp) -> d loss / d logp``
    (or its values), the gradients w.r.t. hidden, weight and bias."""
    h, w = hidden.detach().double(), weight.detach().double()
    b = bias.detach().double() if bias is not None else None
    live = ids != IGNORE
    safe = torch.where(live, ids, torch.zeros_like(ids))
    blocks = [slice(lo, min(lo + 1024, h.size(0))) for lo in range(0, h.size(0), 1024)]

    def scaled(rows):
        z = h[rows] @ w.t()
        return (z if b is None else z + b).div_(temperature)

    logp, lse = torch.empty_like(h[:, 0]), torch.empty_like(h[:, 0])
    for rows in blocks:
        z = scaled(rows)
        lse[rows] = torch.logsumexp(z, 1)
        logp[rows] = torch.where(live[rows], z.gather(1, safe[rows, None])[:, 0] - lse[rows], torch.zeros_like(lse[rows]))
        del z
    if upstream is None:
        return logp, None
    g = upstream(logp) if callable(upstream) else upstream.double()
    g = torch.where(live, g, torch.zeros_like(g)) / temperature
    dh, dw, db = torch.empty_like(h), torch.zeros_like(w), torch.zeros_like(w[:, 0])
    for rows in blocks:
        dz = scaled(rows).sub_(lse[rows, None]).exp_().mul_(-g[rows, None])
        dz.scatter_add_(1, safe[rows, None], g[rows, None])
        dh[rows] = dz @ w
        dw.addmm_(dz.t(), h[rows])
        db += dz.sum(0)
        del dz
    return logp, (dh, dw, db)


def _exact_grpo(cur, old, ref, rewards, mask, group, beta, clip=0.2):
    """float64 ``(loss, policy, kl)`` of the masked mean of the clipped ratio terms and k3 KL."""
    r = rewards.double().view(-1, group)
    std = ((r * r).mean(1, keepdim=True) - r.mean(1, keepdim=True) ** 2).clamp_min(1e-12).sqrt()
    adv = ((r - r.mean(1, keepdim=True)) / std).view(-1, 1)
    keep, zero = mask.bool(), torch.zeros_like(cur)
    ratio = torch.exp(torch.where(keep, cur - old.double(), zero))
    policy = -torch.minimum(ratio * adv, ratio.clamp(1 - clip, 1 + clip) * adv)
    diff = torch.where(keep, ref.double() - cur, zero)
    count = keep.sum()
    policy = torch.where(keep, policy, zero).sum() / count
    kl = torch.where(keep, diff.exp() - diff - 1, zero).sum() / count
    return policy + beta * kl, policy, kl


def exact(case, seed):
    """What ``run`` returns for these inputs, by plain torch in float64."""
    state = prepare(case, seed)
    path = case["path"]
    if path.startswith("logits"):
        def selected(logits, ids):
            return torch.cat([z.double().gather(1, i[:, None])[:, 0] - torch.logsumexp(z.double(), 1)
                              for z, i in zip(logits.split(512), ids.split(512))])

        logits, ids = state["logits"].detach().view(-1, case["vocab"]), state["ids"].reshape(-1)
        cur = selected(logits, ids)
        if path == "logits_logp":
            return cur
        cur.requires_grad_(True)
        ref = selected(state["ref"].view(-1, case["vocab"]), ids)
        shape = state["ids"].shape
        out = _exact_grpo(cur.view(shape), state["old"], ref.view(shape), state["rewards"], state["mask"],
                          case["group"], 0.04)
        g, = torch.autograd.grad(out[0], [cur])
        grad = torch.empty(logits.shape, device=logits.device, dtype=torch.float64)
        for lo in range(0, len(cur), 512):
            rows = slice(lo, lo + 512)
            dz = torch.softmax(logits[rows].double(), 1).mul_(-g[rows, None])
            grad[rows] = dz.scatter_add_(1, ids[rows, None], g[rows, None])
        return (*(x.detach() for x in out), grad.view(state["logits"].shape))
    if path == "score":
        args = (state["ids"], case["temperature"])
        logp = _exact_head(state["hidden"], state["weight"], state["bias"], *args)[0]
        if not case["reference"]:
            return logp
        return logp, _exact_head(state["hidden"], state["ref_weight"], state["ref_bias"], *args)[0]
    if path == "train":
        x = state["hidden"].detach().double()
        if case["norm"]:
            gain = state["gain"].detach().double()
            rstd = (x.square().mean(1, keepdim=True) + 1e-6).rsqrt()
            y = x * rstd * gain
        else:
            y = x
        logp, (dh, dw, db) = _exact_head(y, state["weight"], state["bias"], state["ids"], case["temperature"],
                                         state["upstream"])
        grads = [dh]
        if case["norm"]:
            d = dh * gain
            grads[0] = rstd * (d - x * rstd * rstd * (d * x).mean(1, keepdim=True))
        if not case["main_grad"]:
            grads.append(dw)
        if case["norm"]:
            grads.append((dh * x * rstd).sum(0))
        if case["bias"]:
            grads.append(db)
        return (logp, *grads, dw if case["main_grad"] else None)
    shape = state["ids"].shape
    ids = torch.where(state["mask"], state["ids"], torch.full_like(state["ids"], IGNORE)).view(-1)
    values = []

    def upstream(logp):
        cur = logp.detach().view(shape).requires_grad_(True)
        out = _exact_grpo(cur, state["old"], state["ref"], state["rewards"], state["mask"], case["group"], 0.04)
        values.extend(x.detach() for x in out)
        return torch.autograd.grad(out[0], [cur])[0].view(-1)

    logp, (dh, dw, db) = _exact_head(state["hidden"].view(-1, case["hidden"]), state["head"].weight, state["bias"],
                                     ids, case["temperature"], upstream)
    return (*values, logp.view(shape), dh.view(state["hidden"].shape), dw) + ((db,) if case["bias"] else ())
