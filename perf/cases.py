"""What this framework is timed on: the losses of a language-model head, through
the public entry points and over the sizes a training or evaluation program
calls them with.

Kinds of case (``case["kind"]``):

  ce      ``tiled_linear_cross_entropy``, forward and backward
  eval    the same without gradients, per-token losses (an evaluation pass)
  layer   ``VocabParallelLinear.parallel_cross_entropy`` with its default, per-token
          losses; the caller multiplies them by token weights and sums, and the
          backward gets one upstream gradient per token
  masked  ``masked_token_loss``: token weights, output multiplier, mask token
          excluded from the softmax
  drafter ``dflash_token_loss`` over a boolean supervision mask, frozen head
  kl      ``frozen_linear_kl`` between two frozen heads
  topk    ``frozen_linear_ce_topk``: loss, label probability, exact top-k logits
  soft    ``streaming_soft_embedding`` (forward only)

``rows`` is the number of tokens handed in, ``loss_rows`` how many of them bear
a loss (the others carry the ignore label); ``hidden`` and ``vocab`` are the
head's.
"""

from __future__ import annotations

import math

import torch

from turbo_dllm_amd.dflash_kl import frozen_linear_kl
from turbo_dllm_amd.dflash_linear_topk import frozen_linear_ce_topk
from turbo_dllm_amd.layers import VocabParallelLinear
from turbo_dllm_amd.loss import dflash_token_loss, masked_token_loss
from turbo_dllm_amd.streaming_soft_embedding import streaming_soft_embedding
from turbo_dllm_amd.tiled_linear_cross_entropy import tiled_linear_cross_entropy

IGNORE = -100
_DTYPES = {"bf16": torch.bfloat16, "f16": torch.float16, "f32": torch.float32}


def _case(kind, rows, hidden, vocab, *, loss_rows=None, dtype="bf16", reduction="mean",
          softcap=0.0, exclude=False, bias=False, dim_first=False, trainable=True, zipf=False,
          samples=1, top_k=0, multiplier=1.0, name=None):
    case = {
        "kind": kind, "rows": rows, "loss_rows": rows if loss_rows is None else loss_rows,
        "hidden": hidden, "vocab": vocab, "dtype": dtype, "reduction": reduction,
        "softcap": softcap, "exclude": exclude, "bias": bias, "dim_first": dim_first,
        "trainable": trainable, "zipf": zipf, "samples": samples, "top_k": top_k,
        "multiplier": multiplier,
    }
    return case if name is None else {"name": name, **case}


def listed():
    return [
        # one short sequence through a small head: launches and host work are the time
        _case("ce", 64, 1024, 32000, name="one_short_sequence"),
        # a small model's step, about half of its tokens masked
        _case("ce", 2048, 1024, 32000, loss_rows=1036, name="small_head"),
        # 32000 words and three added special tokens, the mask token the last of them and
        # excluded from the softmax: no vocabulary of whole tiles
        _case("ce", 4096, 2048, 32003, loss_rows=2741, reduction="sum", exclude=True,
              name="odd_vocabulary"),
        # float32 training (the operator's default dtype) of a small head
        _case("ce", 1024, 1024, 32000, dtype="f32", name="float32_head"),
        # evaluation: per-token losses of masked sequences, no gradients
        _case("eval", 8192, 4096, 151936, loss_rows=6357, reduction="none", name="evaluation"),
        # the loss call of a model's head layer: per-token losses of a fully masked half
        _case("layer", 16384, 4096, 151936, reduction="none", name="layer_per_token"),
        # the headline step: every row of a clean + noisy pair of halves bears loss
        _case("ce", 32768, 4096, 151936, name="block_diffusion_all_rows"),
        # masked-token loss of a large soft-capped head, half of the rows masked
        _case("masked", 16384, 3840, 262144, loss_rows=8212, softcap=30.0, exclude=True,
              multiplier=0.5, name="softcap_masked_loss"),
        # a drafter under a frozen head, 5 % of packed tokens supervised, Zipf labels
        _case("drafter", 32768, 4096, 151936, loss_rows=1610, trainable=False, zipf=True,
              samples=64, name="sparse_drafter"),
        # distillation: forward KL of a teacher head against a draft head, both frozen
        _case("kl", 8192, 4096, 151936, trainable=False, name="frozen_kl"),
        # confidence-weighted drafter losses: loss, label probability and top logits
        _case("topk", 8192, 4096, 151936, trainable=False, top_k=16, name="loss_and_top_k"),
        # soft token embeddings of a soft-capped head (self-conditioning)
        _case("soft", 8192, 3840, 262144, softcap=30.0, trainable=False, name="soft_embedding"),
    ]


_LARGEST_FLOPS = 6.0 * 32768 * 4096 * 151936
# float32 runs at a fraction of the 16-bit rate: its drawn cases stay in proportion
_LARGEST_F32_FLOPS = 6.0 * 2048 * 1024 * 32000


def _spread(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def draw(rng):
    kind = rng.choice(["ce", "ce", "ce", "eval", "layer", "masked", "drafter", "kl", "topk", "soft"])
    dtype = "bf16"
    if kind in ("ce", "eval", "layer", "masked"):
        dtype = rng.choice(["bf16"] * 8 + ["f16", "f32"])
    # head widths are multiples of 64 in nearly every model; vocabularies are often padded
    # to one, and otherwise whatever the tokenizer gives
    hidden = 64 * _spread(rng, 8, 64)
    if rng.random() < 0.1:
        hidden -= 8 * rng.randint(1, 7)
    vocab = _spread(rng, 16384, 262144)
    if rng.random() < 0.7:
        vocab = (vocab + 63) // 64 * 64
    rows = _spread(rng, 64, 32768)
    softcap = rng.choice([0.0, 0.0, 0.0, 30.0])
    if kind == "soft":
        softcap = rng.choice([0.0, 30.0])
    share = rng.choice([1.0, rng.uniform(0.05, 1.0)])
    samples = 1
    if kind == "drafter":
        samples = rng.choice([1, 4, 16])
        rows = max(rows // samples, 4) * samples
    limit = _LARGEST_F32_FLOPS if dtype == "f32" else _LARGEST_FLOPS
    # (two frozen heads, or statistics and top-k, cost more time per useful operation)
    limit *= 0.5
    while 6.0 * rows * hidden * vocab > limit:
        rows = max(rows // 2 // samples, 4) * samples
    whole = kind in ("kl", "topk", "soft")
    return _case(
        kind, rows, hidden, vocab,
        loss_rows=rows if whole else max(1, int(rows * share)),
        dtype=dtype,
        reduction="none" if kind in ("eval", "layer") else rng.choice(["mean", "mean", "sum"]),
        softcap=softcap,
        exclude=kind in ("ce", "eval", "masked") and rng.random() < 0.3,
        bias=kind in ("ce", "layer") and rng.random() < 0.1,
        dim_first=kind == "ce" and rng.random() < 0.1,
        trainable=kind not in ("drafter", "kl", "topk", "soft") and rng.random() < 0.8,
        zipf=rng.random() < 0.3, samples=samples,
        top_k=rng.choice([1, 8, 16, 64]) if kind == "topk" else 0,
        multiplier=0.5 if kind == "masked" else 1.0,
    )


# ------------------------------------------------------------------ inputs --
def _labels(case, gen, device):
    """Target ids (uniform, or Zipf with exponent 1.1), never the excluded last id;
    exactly ``loss_rows`` of them kept, the rest set to the ignore label."""
    n, v = case["rows"], case["vocab"] - 1
    if case["zipf"]:
        cdf = torch.arange(1, v + 1, dtype=torch.float64, device=device).pow(-1.1).cumsum(0)
        u = torch.rand(n, generator=gen, dtype=torch.float64, device=device) * cdf[-1]
        labels = torch.searchsorted(cdf, u).clamp_(max=v - 1)
    else:
        labels = torch.randint(0, v, (n,), generator=gen, device=device)
    keep = torch.zeros(n, dtype=torch.bool, device=device)
    order = torch.rand(n, generator=gen, device=device).argsort()
    keep[order[:case["loss_rows"]]] = True
    return labels, keep


def _hidden_for(labels, weight, gen, n, h, device, logit=8.0):
    """Hidden states of a model in training: noise, and a component along the label's
    head row that raises its logit by about ``logit``."""
    hidden = torch.randn(n, h, generator=gen, device=device)
    for lo in range(0, n, 4096):
        rows = weight[labels[lo:lo + 4096]].float()
        hidden[lo:lo + 4096] += rows * (logit / rows.pow(2).sum(1, keepdim=True))
    return hidden


def _head(weight, bias, trainable):
    with torch.device("meta"):
        head = VocabParallelLinear(weight.shape[1], weight.shape[0], bias=bias is not None)
    head.weight = torch.nn.Parameter(weight, requires_grad=trainable)
    if bias is not None:
        head.bias = torch.nn.Parameter(bias, requires_grad=trainable)
    return head


def prepare(case, seed):
    device = torch.device("cuda")
    gen = torch.Generator(device=device).manual_seed(int(seed))
    n, h, v = case["rows"], case["hidden"], case["vocab"]
    dtype = _DTYPES[case["dtype"]]
    weight = torch.empty(v, h, dtype=dtype, device=device)
    for lo in range(0, v, 32768):
        part = weight[lo:lo + 32768]
        part.copy_(torch.randn(part.shape, generator=gen, device=device) * 0.02)
    labels, keep = _labels(case, gen, device)
    hidden = _hidden_for(labels, weight, gen, n, h, device)
    state = {"case": case, "labels": labels}
    if case["kind"] in ("ce", "eval", "layer", "masked"):
        state["labels"] = torch.where(keep, labels, torch.full_like(labels, IGNORE))
        state["token_weights"] = torch.rand(n, generator=gen, device=device) + 0.5
    if case["kind"] == "drafter":
        b = case["samples"]
        hidden = hidden.reshape(b, n // b, h)
        state["labels"] = labels.reshape(b, n // b)
        state["mask"] = keep.reshape(b, n // b)
        state["token_weights"] = torch.rand(b, n // b, generator=gen, device=device) + 0.5
        state["counts"] = state["mask"].sum(1).float()
    if case["kind"] == "kl":
        # the draft head is near the teacher's, and the draft's hidden states near its own
        teacher_weight = weight.clone()
        for lo in range(0, v, 32768):
            part = weight[lo:lo + 32768]
            part.add_((torch.randn(part.shape, generator=gen, device=device) * 0.01).to(dtype))
        state["teacher_hidden"] = hidden.to(dtype)
        state["teacher_weight"] = teacher_weight
        hidden = hidden + 0.5 * torch.randn(hidden.shape, generator=gen, device=device)
        state["upstream"] = torch.rand(n, generator=gen, device=device) / n
    if case["kind"] == "topk":
        state["upstream"] = torch.rand(3, n, generator=gen, device=device) / n
    hidden = hidden.to(dtype)
    bias = None
    if case["bias"]:
        bias = (torch.randn(v, generator=gen, device=device) * 0.1).to(dtype)
    if case["dim_first"]:
        weight = weight.t().contiguous()
    grad = case["kind"] not in ("eval", "soft")
    state["hidden"] = hidden.requires_grad_(grad)
    if case["kind"] in ("layer", "masked", "drafter"):
        state["head"] = _head(weight, bias, case["trainable"])
    else:
        state["weight"] = weight.requires_grad_(grad and case["trainable"])
        state["bias"] = None if bias is None else bias.requires_grad_(grad and case["trainable"])
    return state


# -------------------------------------------------------------------- pass --
def _grads(loss, leaves):
    """The backward of a training step, and the gradients it leaves."""
    leaves = [t for t in leaves if t is not None and t.requires_grad]
    for t in leaves:
        t.grad = None
    loss.backward()
    return [t.grad for t in leaves]


def run(state):
    case = state["case"]
    kind, hidden, labels = case["kind"], state["hidden"], state["labels"]
    exclude = case["vocab"] - 1 if case["exclude"] else None
    softcap = case["softcap"] or None
    if kind in ("ce", "eval"):
        def loss_of():
            return tiled_linear_cross_entropy(
                hidden, state["weight"], labels, bias=state["bias"],
                reduction=case["reduction"], exclude_index=exclude, logit_softcap=softcap,
                dtype=hidden.dtype,
                weight_layout="dim_first" if case["dim_first"] else "vocab_first")
        if kind == "eval":
            with torch.no_grad():
                return loss_of()
        loss = loss_of()
        return [loss.detach(), *_grads(loss, (hidden, state["weight"], state["bias"]))]
    if kind == "layer":
        head = state["head"]
        losses = head.parallel_cross_entropy(hidden, labels, logit_softcap=softcap)
        total = (losses * state["token_weights"]).sum() / case["loss_rows"]
        return [losses.detach(), *_grads(total, (hidden, head.weight, head.bias))]
    if kind == "masked":
        head = state["head"]
        loss = masked_token_loss(
            hidden, labels, state["token_weights"], head,
            valid_token_count=float(case["loss_rows"]), mask_token_id=case["vocab"] - 1,
            exclude_mask_token=case["exclude"], output_multiplier=case["multiplier"],
            logit_softcap=softcap)
        return [loss.detach(), *_grads(loss, (hidden, head.weight))]
    if kind == "drafter":
        loss = dflash_token_loss(
            hidden, labels, state["mask"], state["token_weights"], state["head"],
            loss_kind="paper_ce", normalization_count=state["counts"], logit_softcap=softcap)
        return [loss.detach(), *_grads(loss, (hidden, state["head"].weight))]
    if kind == "kl":
        losses = frozen_linear_kl(hidden, state["weight"], state["teacher_hidden"],
                                  state["teacher_weight"], logit_softcap=softcap)
        return [losses.detach(), *_grads((losses * state["upstream"]).sum(), (hidden,))]
    if kind == "topk":
        loss, probability, values, ids = frozen_linear_ce_topk(
            hidden, state["weight"], labels, top_k=case["top_k"], logit_softcap=softcap)
        up = state["upstream"]
        total = (loss * up[0] + probability * up[1] + values.mean(1) * up[2]).sum()
        return [loss.detach(), probability.detach(), values.detach(), ids,
                *_grads(total, (hidden,))]
    return streaming_soft_embedding(hidden, state["weight"], row_chunk_size=1024,
                                    vocab_chunk_size=32768, logit_softcap=softcap,
                                    embedding_scale=math.sqrt(case["hidden"]))


# --------------------------------------------------------------- yardstick --
def work(case):
    m, n, h, v = case["loss_rows"], case["rows"], case["hidden"], case["vocab"]
    es = 4 if case["dtype"] == "f32" else 2
    kind = case["kind"]
    contractions = {"eval": 1, "kl": 3, "topk": 2, "soft": 2}.get(
        kind, 3 if case["trainable"] else 2)
    heads = 2 if kind == "kl" else 1
    bytes_ = heads * (m * h + v * h) * es + 8 * n          # rows, head, labels
    if kind == "eval":
        bytes_ += 4 * n
    else:
        bytes_ += n * h * es                               # grad_hidden or the output
        if case["trainable"]:
            bytes_ += v * h * es
    if kind in ("layer", "masked", "drafter", "kl", "topk"):
        bytes_ += 8 * n                                    # per-token factors and losses
    if kind == "topk":
        bytes_ += 12 * n * case["top_k"]
    return {"bytes": bytes_, "flops": 2.0 * contractions * m * h * v}


def tolerance(case):
    # About four times what two correct paths differ by.  16-bit: gradients are sums over
    # softmax entries rounded to the dtype, and are rounded once themselves (against
    # float64 and between the two ways of forming them: 2e-3 to 3.7e-3 in the 2-norm, up
    # to 0.16 for a single entry of grad_weight beside its root mean square).  float32:
    # 3.3e-6 and 2.6e-5 against float64.  "differ": near-ties among the top-k ids.
    if case["dtype"] == "f32":
        return {"rel": 1.3e-5, "max": 1e-4, "differ": 0.0}
    return {"rel": 1.4e-2, "max": 0.6, "differ": 1e-3}
