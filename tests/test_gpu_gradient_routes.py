"""Which calls leave their gradients in the forward, and what that costs in exactness.

An entry rounded to bf16 is off by 2^-7 / sqrt(12) * sqrt(3 / (8 ln 2)) = 1.66e-3 relative
(root mean square, mantissas spread evenly over a binade).  The recomputing backward rounds
the logit gradients and the result, sqrt(2) * 1.66e-3 = 2.35e-3 in the 2-norm; gradients
formed in the forward also round the hidden rows times their row factor on the way to
grad_weight, sqrt(3) * 1.66e-3 = 2.87e-3.  Calls that must be as exact as the recomputing
backward are held to the middle of the two, 2.6e-3."""

import pytest
import torch

import linear_ce_oracle as oracle
from turbo_dllm_amd import _lib, options
from turbo_dllm_amd.dflash_kl import frozen_linear_kl
from turbo_dllm_amd.dflash_linear_topk import frozen_linear_ce_topk
from turbo_dllm_amd.streaming_soft_embedding import streaming_soft_embedding
from turbo_dllm_amd.tiled_linear_cross_entropy import tiled_linear_cross_entropy

pytestmark = pytest.mark.gpu

TWO_ROUNDINGS = 2.6e-3


def operands(dev, m, h, v, seed=3):
    gen = torch.Generator().manual_seed(seed)
    weight = (torch.randn(v, h, generator=gen) * 0.05).bfloat16().to(dev)
    labels = torch.randint(0, v, (m,), generator=gen).to(dev)
    hidden = torch.randn(m, h, generator=gen).to(dev)
    hidden = (hidden + weight[labels].float() * (8.0 / (0.05 ** 2 * h))).bfloat16()
    return hidden, weight, labels, torch.rand(m, generator=gen).to(dev) + 0.5


def step(hidden, weight, labels, upstream, reduction, trainable=True, **kw):
    x = hidden.clone().requires_grad_(True)
    w = weight.clone().requires_grad_(trainable)
    loss = tiled_linear_cross_entropy(x, w, labels, reduction=reduction, dtype=torch.bfloat16, **kw)
    (loss * upstream).sum().backward() if reduction == "none" else loss.backward()
    torch.cuda.synchronize()
    return loss.detach(), x.grad, w.grad


def exact_grad_weight(hidden, weight, labels, row_factors, rows=1024):
    """sum_r factor_r (softmax - onehot)_r hidden_r in float64."""
    w = weight.double()
    out = torch.zeros_like(w)
    for lo in range(0, hidden.shape[0], rows):
        x = hidden[lo:lo + rows].double()
        g = (x @ w.t()).softmax(1)
        g[torch.arange(len(x), device=g.device), labels[lo:lo + rows]] -= 1.0
        out += (g * row_factors[lo:lo + rows, None]).t() @ x
    return out


def relative_norm(got, want):
    return float((got.double() - want).norm() / want.norm())


@pytest.mark.parametrize("trainable", [True, False])
@pytest.mark.parametrize("reduction", ["mean", "sum", "none"])
@pytest.mark.parametrize("m,h,v,kw", [
    (700, 256, 50257, {}),
    (1030, 320, 32003, dict(logit_softcap=30.0, exclude_index=32002)),
])
def test_ragged_vocabularies_recompute(gpu_device, m, h, v, kw, reduction, trainable):
    print("[case]", m, h, v, reduction, trainable, kw, flush=True)
    hidden, weight, labels, up = operands(gpu_device, m, h, v - 1)
    weight = torch.cat([weight, weight[:1]])
    with _lib.kernel_profile() as prof:
        got = step(hidden, weight, labels, up, reduction, trainable, **kw)
    assert prof.launches["exp_logits_panel"] == 0 and prof.launches["forward_stats"] > 0
    with options.gradient_mode("recompute"):
        want = step(hidden, weight, labels, up, reduction, trainable, **kw)
    for a, b in zip(got, want):
        assert (a is None and b is None) or torch.equal(a, b)
    if trainable and not kw and reduction != "none":
        factor = torch.full((m,), 1.0 / m if reduction == "mean" else 1.0, device=gpu_device)
        error = relative_norm(got[2], exact_grad_weight(hidden, weight, labels, factor.double()))
        print("[case] grad_weight error", error, flush=True)
        assert error <= TWO_ROUNDINGS


@pytest.mark.parametrize("softcap", [None, 30.0])
def test_ragged_soft_embedding_rounds_normalised_probabilities(gpu_device, softcap):
    hidden, weight, _, _ = operands(gpu_device, 300, 256, 3001)
    with _lib.kernel_profile() as prof:
        got = streaming_soft_embedding(hidden, weight, row_chunk_size=64, vocab_chunk_size=1024,
                                       logit_softcap=softcap)
    assert prof.launches["exp_logits_panel"] == 0 and prof.launches["forward_stats"] > 0
    z = hidden.double() @ weight.double().t()
    if softcap is not None:
        z = softcap * torch.tanh(z / softcap)
    assert relative_norm(got, z.softmax(1) @ weight.double()) <= TWO_ROUNDINGS


# 10240 rows over V = 151936: two blocks of the default panel of 2.5 GiB
BLOCKED = (10240, 64, 151936)


def test_rows_beyond_the_default_panel_hold_no_panel_until_the_backward(gpu_device):
    """Between forward and backward, where a model's activations are live, only the float32
    gradients may be held; the panel of the step (3.1 GB in one block) is released."""
    m, h, v = BLOCKED
    hidden, weight, labels, _ = operands(gpu_device, m, h, v)
    x, w = hidden.requires_grad_(True), weight.requires_grad_(True)
    torch.cuda.synchronize()
    before = torch.cuda.memory_allocated()
    with _lib.kernel_profile() as prof:
        loss = tiled_linear_cross_entropy(x, w, labels, reduction="mean", dtype=torch.bfloat16)
    held = torch.cuda.memory_allocated() - before
    gradients = 4 * h * (m + v)
    print("[case] held", held, "float32 gradients", gradients, flush=True)
    assert prof.launches["grad_weight_gemm"] == 2
    assert held <= gradients + (1 << 20)
    loss.backward()
    torch.cuda.synchronize()
    ones = torch.full((m,), 1.0 / m, dtype=torch.float64, device=gpu_device)
    # (gradients formed in the forward: three roundings of grad_weight, 2.87e-3, and 8 % for the
    # spread of one sample)
    assert relative_norm(w.grad, exact_grad_weight(hidden.detach(), weight.detach(), labels, ones)) <= 3.1e-3


def test_per_token_losses_beyond_one_block_recompute(gpu_device):
    m, h, v = BLOCKED
    hidden, weight, labels, up = operands(gpu_device, m, h, v)
    with _lib.kernel_profile() as prof:
        got = step(hidden, weight, labels, up, "none")
    assert prof.launches["exp_logits_panel"] == 0
    with options.gradient_mode("recompute"):
        want = step(hidden, weight, labels, up, "none")
    for a, b in zip(got, want):
        assert torch.equal(a, b)
    error = relative_norm(got[2], exact_grad_weight(hidden, weight, labels, up.double()))
    print("[case] grad_weight error", error, flush=True)
    assert error <= TWO_ROUNDINGS


# KL and CE with top-k form their gradients in the forward over any vocabulary: the last K
# slab of the contraction over it comes from a zero-padded copy of the head's last rows
RAGGED = [(1, 64, 2), (65, 64, 63), (130, 128, 65), (257, 192, 191), (300, 256, 4099)]


@pytest.mark.parametrize("softcap", [None, 20.0])
@pytest.mark.parametrize("m,h,v", RAGGED)
def test_ragged_kl_gradient_in_the_forward(gpu_device, m, h, v, softcap):
    """Loss and gradient at the operator's bars for bf16 (rtol 2e-2 / atol 1e-3, relative
    max-norm 2e-2 of the float64 oracle)."""
    print("[case]", m, h, v, softcap, flush=True)
    gen = torch.Generator().manual_seed(m + v)
    cpu = [(torch.randn(n, h, generator=gen) * std).bfloat16()
           for n, std in ((m, 1.0), (v, 0.2), (m, 1.0), (v, 0.2))]
    ops = [t.to(gpu_device) for t in cpu]
    up = torch.rand(m, generator=gen) + 0.1
    x = ops[0].clone().requires_grad_(True)
    with _lib.kernel_profile() as prof:
        losses = frozen_linear_kl(x, *ops[1:], logit_softcap=softcap)
    assert prof.launches["grad_hidden_gemm"] == 1
    losses.backward(up.to(gpu_device))
    torch.cuda.synchronize()
    want = oracle.dense_frozen_kl(*cpu, logit_softcap=softcap)
    torch.testing.assert_close(losses.detach().cpu().double(), want, rtol=2e-2, atol=1e-3)
    grad = oracle.dense_frozen_kl_grad(*cpu, up, logit_softcap=softcap)
    assert oracle.relative_max_error(x.grad, grad) <= 2e-2


@pytest.mark.parametrize("softcap", [None, 20.0])
@pytest.mark.parametrize("m,h,v", RAGGED)
def test_ragged_top_k_gradient_in_the_forward(gpu_device, m, h, v, softcap):
    print("[case]", m, h, v, softcap, flush=True)
    k = min(v, 7)
    gen = torch.Generator().manual_seed(m + v)
    hidden = torch.randn(m, h, generator=gen).bfloat16()
    weight = (torch.randn(v, h, generator=gen) * 0.2).bfloat16()
    labels = torch.randint(0, v, (m,), generator=gen)
    up = torch.rand(3, m, generator=gen)
    x = hidden.to(gpu_device).requires_grad_(True)
    with _lib.kernel_profile() as prof:
        loss, prob, values, ids = frozen_linear_ce_topk(
            x, weight.to(gpu_device), labels.to(gpu_device), top_k=k, logit_softcap=softcap)
    assert prof.launches["grad_hidden_gemm"] == 1
    g = up.to(gpu_device)
    (loss * g[0] + prob * g[1] + values.mean(1) * g[2]).sum().backward()
    torch.cuda.synchronize()
    z = hidden.double() @ weight.double().t()
    z = z if softcap is None else softcap * torch.tanh(z / softcap)
    want = torch.logsumexp(z, 1) - z.gather(1, labels[:, None])[:, 0]
    torch.testing.assert_close(loss.detach().cpu().double(), want, rtol=1e-4, atol=1e-4)
    grad = oracle.dense_ce_topk_grad(hidden, weight, labels, ids.cpu(), up[0], up[1],
                                     up[2][:, None].expand(m, k) / k, logit_softcap=softcap)
    assert oracle.relative_max_error(x.grad, grad) <= 2e-2


def test_ragged_objectives_in_several_blocks_of_rows(gpu_device):
    """V = 150001, 9000 rows: two blocks of the 2.5 GiB panel for each objective.  Gradients
    against float64 in the 2-norm: entries rounded twice at most (when written, and where a
    maximum moved) and the result once, 2.87e-3, and 8 % for the spread of one sample."""
    m, h, v = 9000, 64, 150001
    hidden, weight, labels, up = operands(gpu_device, m, h, v)
    teacher, teacher_weight, _, _ = operands(gpu_device, m, h, v, seed=4)
    x = hidden.clone().requires_grad_(True)
    with _lib.kernel_profile() as prof:
        losses = frozen_linear_kl(x, weight, teacher, teacher_weight)
    assert prof.launches["grad_hidden_gemm"] == 2
    losses.backward(up)
    y = hidden.clone().requires_grad_(True)
    with _lib.kernel_profile() as prof:
        ce, _, _, _ = frozen_linear_ce_topk(y, weight, labels, top_k=4)
    assert prof.launches["grad_hidden_gemm"] == 2
    ce.backward(up)
    w, tw = weight.double(), teacher_weight.double()
    wants = [[], [], [], []]
    for lo in range(0, m, 500):
        part = slice(lo, lo + 500)
        draft, factor = (hidden[part].double() @ w.t()).log_softmax(1), up[part, None].double()
        target = (teacher[part].double() @ tw.t()).log_softmax(1)
        wants[0].append((target.exp() * (target - draft)).sum(1))
        wants[1].append(((draft.exp() - target.exp()) * factor) @ w)
        wants[2].append(-draft.gather(1, labels[part, None])[:, 0])
        wants[3].append(factor * (draft.exp() @ w - w[labels[part]]))
    kl, kl_grad, nll, nll_grad = (torch.cat(t) for t in wants)
    for got, want in ((losses, kl), (ce, nll)):
        torch.testing.assert_close(got.detach().double(), want, rtol=1e-3, atol=1e-3)
    for got, want in ((x.grad, kl_grad), (y.grad, nll_grad)):
        error = relative_norm(got, want)
        print("[case] gradient error", error, flush=True)
        assert error <= 3.1e-3
