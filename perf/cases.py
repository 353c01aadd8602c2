"""The calls whose speed is followed, over the range that they are made in.

Each case is one call of the public API as a training or an evaluation loop
makes it: the loss of given logits (``vocab_parallel_cross_entropy`` forward
and backward, its per-token form without a gradient, one tensor-parallel
rank's shard through the C entries), and the fused LM head + loss
(``lmhead_vocab_parallel_cross_entropy`` forward and backward, and without a
gradient). Inputs lie on the GPU; a pass returns the loss and the gradients.

The loss's in-place form runs the kernels of the out-of-place one with the
destination moved; it would consume its inputs, so passes here keep the
default and get the gradient in a new tensor.
"""

import math
import pathlib
import sys

import torch

sys.path.insert(0, str(pathlib.Path(__file__).resolve().parent.parent / "nano-megatron_amd"))

import nmce  # noqa: E402
from nmce import _lib  # noqa: E402

_DTYPES = {"bf16": torch.bfloat16, "f32": torch.float32}


def listed():
    return [
        # The smallest call: a fine-tuning micro-batch of a few dozen tokens,
        # where launches and the host's share count.
        _ce("ce_small", "bf16", 1, 64, 50304),
        # fp32 logits of a small batch (a model run without autocast).
        _ce("ce_f32", "f32", 4, 256, 32000),
        # The ordinary bf16 training batch at a padded GPT-2 vocabulary.
        _ce("ce_bf16", "bf16", 8, 2048, 50304),
        # The same vocabulary unpadded: rows of an odd number of columns, which
        # start off the 16-byte grid.
        _ce("ce_ragged", "bf16", 2, 2048, 50257),
        # A whole 128256-entry vocabulary on one GPU: the widest rows in use.
        _ce("ce_wide", "bf16", 4, 2048, 128256),
        # Evaluation: the per-token loss of held-out text, no gradient.
        dict(name="ce_eval", kind="ce_eval", dtype="bf16", b=8, s=1024, v=50304),
        # One rank of a tensor-parallel pair (the upper half of 128256 ids):
        # local statistics, the merge with the other rank's, the gradient.
        dict(name="tp_shard", kind="tp_shard", dtype="bf16", b=4, s=4096, v=64128),
        # The fused head of a small model (GPT-2 width) at one short sequence.
        _head("head_small", 1, 512, 768, 50304),
        # Odd everywhere: 2103 tokens, a width of 25 heads of 64, the unpadded
        # vocabulary.
        _head("head_ragged", 3, 701, 1600, 50257),
        # One long sequence of a large model: the ordinary micro-batch.
        _head("head_micro", 1, 4096, 4096, 128256),
        # The large batch, the most work of a call here.
        _head("head_large", 8, 2048, 4096, 128256),
        # Evaluation with the fused head at the largest vocabulary.
        dict(name="head_eval", kind="head_eval", b=2, s=2048, h=3072, v=256000),
    ]


def _ce(name, dtype, b, s, v):
    return dict(name=name, kind="ce", dtype=dtype, b=b, s=s, v=v)


def _head(name, b, s, h, v):
    return dict(name=name, kind="head", b=b, s=s, h=h, v=v)


_VOCABS = (32000, 50257, 50304, 64128, 100277, 128256, 151936, 256000)


def draw(rng):
    """A case of the listed ones' ranges: tokens and vocabulary spread over
    their logarithm, a known vocabulary half of the time."""
    def spread(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    kind = rng.choice(("ce", "ce", "ce", "ce_eval", "tp_shard", "head", "head", "head",
                       "head_recompute", "head_eval"))
    b = rng.choice((1, 1, 2, 3, 4, 8))
    if kind.startswith("head"):
        most = 16384 * 4096 * 128256  # head_large's tokens x width x vocabulary
        if kind == "head_recompute":
            most = most * 3 // 4      # 8 products' worth of flops against 6
        v = rng.choice(_VOCABS) if rng.random() < 0.5 else spread(8192, 256000)
        h = 64 * rng.randint(8, 64)
        n = min(spread(64, 16384), most // (h * v))
        return dict(kind=kind, b=b, s=max(1, n // b), h=h, v=v)
    dtype = rng.choice(("bf16", "bf16", "f32"))
    v = rng.choice(_VOCABS) if rng.random() < 0.5 else spread(8192, 256000)
    n = min(spread(64, 16384), (4 << 30) // (v * (2 if dtype == "bf16" else 4)))
    return dict(kind=kind, dtype=dtype, b=b, s=max(1, n // b), v=v)


def _targets(b, s, v, g):
    # Token ids as text has them, many small and few large: log-uniform.
    u = torch.rand((b, s), device="cuda", generator=g, dtype=torch.float64)
    return (torch.exp(u * math.log(v + 1.0)) - 1.0).long().clamp_(0, v - 1)


def _logits(dtype, b, s, v, target, g):
    # A model in training: spread-out logits, the target's raised by 0 to 10.
    x = torch.randn((b, s, v), device="cuda", generator=g, dtype=torch.float32).mul_(2.0)
    own = (target >= 0) & (target < v)
    up = torch.rand((b, s), device="cuda", generator=g, dtype=torch.float32).mul_(10.0) * own
    x.scatter_add_(2, target.clamp(0, v - 1).unsqueeze(2), up.unsqueeze(2))
    return x.to(_DTYPES[dtype])


def prepare(case, seed):
    g = torch.Generator(device="cuda").manual_seed(int(seed))
    b, s, v = case["b"], case["s"], case["v"]
    st = dict(kind=case["kind"], v=v, ctx=nmce.ParallelContext.single())
    if case["kind"] in ("ce", "ce_eval"):
        st["target"] = _targets(b, s, v, g)
        st["logits"] = _logits(case["dtype"], b, s, v, st["target"], g)
        st["logits"].requires_grad_(case["kind"] == "ce")
    elif case["kind"] == "tp_shard":
        # Ids of both ranks; this rank holds [v, 2 v). The other rank's row
        # maximum, exp-sum minus one and target logit are what its half gives.
        st["target"] = _targets(b, s, 2 * v, g)
        st["logits"] = _logits(case["dtype"], b, s, v, st["target"] - v, g)
        n = b * s
        stats = torch.zeros((2, 3, n), device="cuda")
        stats[0, 0] = torch.rand(n, device="cuda", generator=g) * 4.0 + 6.0
        stats[0, 1] = torch.rand(n, device="cuda", generator=g) * 200.0 + 20.0
        first = (st["target"].view(-1) < v).float()
        stats[0, 2] = first * (torch.rand(n, device="cuda", generator=g) * 10.0 - 2.0)
        st["stats"] = stats
        st["grad"] = torch.empty_like(st["logits"])
        st["out"] = torch.empty((3, n), device="cuda")
        st["upstream"] = torch.ones(1, device="cuda")
    else:
        h = case["h"]
        train = case["kind"] != "head_eval"
        st["target"] = _targets(b, s, v, g)
        # The final norm's output and an embedding at its initial spread.
        st["hidden"] = torch.randn((b, s, h), device="cuda", generator=g).to(torch.bfloat16)
        st["weight"] = (torch.randn((v, h), device="cuda", generator=g) * 0.02).to(torch.bfloat16)
        st["hidden"].requires_grad_(train)
        st["weight"].requires_grad_(train)
    return st


def run(state):
    kind, v, ctx, target = state["kind"], state["v"], state["ctx"], state["target"]
    if kind == "ce":
        loss = nmce.vocab_parallel_cross_entropy(state["logits"], target, 0, v, ctx)
        (grad,) = torch.autograd.grad(loss, state["logits"])
        return {"loss": loss.detach(), "grad": grad}
    if kind == "ce_eval":
        with torch.no_grad():
            return {"loss": nmce._VocabParallelCrossEntropy.apply(state["logits"], target, 0, v,
                                                                  None, 1)}
    if kind == "tp_shard":
        return _run_shard(state)
    hidden, weight = state["hidden"], state["weight"]
    if kind == "head_eval":
        with torch.no_grad():
            return {"loss": nmce.lmhead_vocab_parallel_cross_entropy(hidden, weight, target, 0, v,
                                                                     ctx)}
    loss = nmce.lmhead_vocab_parallel_cross_entropy(hidden, weight, target, 0, v, ctx,
                                                    one_pass=kind == "head")
    dx, dw = torch.autograd.grad(loss, (hidden, weight))
    return {"loss": loss.detach(), "dhidden": dx, "dweight": dw}


def _run_shard(st):
    """Rank 1 of 2: its statistics, the merge with the gathered ones of rank 0,
    and the gradient of the mean (the sequence around the all-gather)."""
    lib = _lib.load()
    x, grad, out = st["logits"], st["grad"], st["out"]
    v = st["v"]
    n = x.numel() // v
    code = _lib.dtype_code(x.dtype)
    stream = _lib.stream_handle(x.device)
    stats = st["stats"]
    base = stats.data_ptr()
    mine = base + 12 * n
    _lib.check(lib.nmce_ce_fwd_stats(x.data_ptr(), code, n, v, v, st["target"].data_ptr(), v,
                                     mine, mine + 4 * n, mine + 8 * n, stream), "stats")
    _lib.check(lib.nmce_ce_combine(base, base + 4 * n, base + 8 * n, 2, 3 * n, n, out.data_ptr(),
                                   out.data_ptr() + 4 * n, out.data_ptr() + 8 * n, stream),
               "combine")
    _lib.check(lib.nmce_ce_bwd_scaled(x.data_ptr(), grad.data_ptr(), code, n, v, v, v,
                                      st["target"].data_ptr(), v, out.data_ptr() + 4 * n,
                                      out.data_ptr() + 8 * n, st["upstream"].data_ptr(), 0,
                                      float(n), stream), "bwd")
    return {"loss": out[0], "grad": grad}


def work(case):
    n, v = case["b"] * case["s"], case["v"]
    if case["kind"] in ("ce", "ce_eval", "tp_shard"):
        slab = n * v * (2 if case["dtype"] == "bf16" else 4)
        passes = 1 if case["kind"] == "ce_eval" else 2  # read the logits, write the gradient
        return {"bytes": passes * slab + 12 * n, "flops": 0}
    h = case["h"]
    if case["kind"] == "head_eval":
        return {"bytes": 2 * (n + v) * h + 8 * n, "flops": 2 * n * v * h}
    return {"bytes": 4 * (n + v) * h + 8 * n, "flops": 6 * n * v * h}


def tolerance(case):
    # About four times the distance seen from the 64-bit result, and no less
    # than the types give: fp32 sums (1.1e-7 seen for a loss, 2.2e-8 for an
    # fp32 gradient), a gradient rounded once to bf16 (1.1e-3 seen), and for
    # the head's gradients also the exponentials rounded to bf16 before the
    # products (2.1e-3 seen).
    if case["kind"] in ("ce_eval", "head_eval"):
        return {"rel": 1e-6, "max": 1e-5}
    if case["kind"] in ("ce", "tp_shard"):
        return {"rel": 1e-6, "max": 1e-5} if case["dtype"] == "f32" else {"rel": 4e-3, "max": 2e-2}
    return {"rel": 8e-3, "max": 4e-2}


def exact(case, seed):
    st = prepare(case, seed)
    t = st["target"].reshape(-1)
    n, v = t.numel(), case["v"]
    rows = max(1, (1 << 30) // v // 8)  # rows of 64-bit values held at a time: 1 GiB of them
    loss = torch.empty(n, dtype=torch.float64, device="cuda")
    if case["kind"] in ("ce", "ce_eval", "tp_shard"):
        x = st["logits"].detach().view(n, v)
        grad = None if case["kind"] == "ce_eval" else torch.empty((n, v), dtype=torch.float64,
                                                                  device="cuda")
        start = v if case["kind"] == "tp_shard" else 0
        for a in range(0, n, rows):
            z, tt = x[a:a + rows].double(), t[a:a + rows] - start
            own = (tt >= 0) & (tt < v)
            at = tt.clamp(0, v - 1).unsqueeze(1)
            lse = torch.logsumexp(z, 1)
            picked = z.gather(1, at).squeeze(1) * own
            if start:
                other = st["stats"][0, :, a:a + rows].double()
                lse = torch.logaddexp(lse, other[0] + torch.log1p(other[1]))
                picked = picked + other[2]
            loss[a:a + rows] = lse - picked
            if grad is not None:
                p = torch.exp(z - lse.unsqueeze(1))
                p.scatter_add_(1, at, -own.double().unsqueeze(1))
                grad[a:a + rows] = p / n
        if case["kind"] == "ce_eval":
            return {"loss": loss.view(case["b"], case["s"])}
        shape = (case["b"], case["s"], v)
        return {"loss": loss if start else loss.mean(), "grad": grad.view(shape)}
    x, w = st["hidden"].detach().view(n, -1).double(), st["weight"].detach().double()
    train = case["kind"] != "head_eval"
    dx = torch.empty_like(x) if train else None
    dw = torch.zeros_like(w) if train else None
    for a in range(0, n, rows):
        z, at = x[a:a + rows] @ w.t(), t[a:a + rows].unsqueeze(1)
        lse = torch.logsumexp(z, 1)
        loss[a:a + rows] = lse - z.gather(1, at).squeeze(1)
        if train:
            z.sub_(lse.unsqueeze(1)).exp_()
            z.scatter_add_(1, at, torch.full_like(at, -1, dtype=torch.float64))
            z.div_(n)
            dx[a:a + rows] = z @ w
            dw.addmm_(z.t(), x[a:a + rows])
    if not train:
        return {"loss": loss.mean()}
    return {"loss": loss.mean(), "dhidden": dx.view(st["hidden"].shape), "dweight": dw}
