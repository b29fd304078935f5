"""The k largest logits found from exponentiated ones (rows x words >= 2^25): exact on exactly
representable logits whatever settles them (the selection, its pruning, the scan that rows of
many ties fall back to), and close to float64 otherwise."""

import pytest
import torch

from turbo_dllm_amd.dflash_linear_topk import frozen_linear_ce_topk

pytestmark = pytest.mark.gpu


def run(hidden, weight, labels, k, cap=None, up=None):
    x = hidden.clone().requires_grad_()
    loss, prob, values, ids = frozen_linear_ce_topk(x, weight, labels, top_k=k, logit_softcap=cap)
    if up is not None:
        (loss * up[0] + prob * up[1] + values.mean(1) * up[2]).sum().backward()
    return loss.detach(), prob.detach(), values.detach(), ids, x.grad


def exact(hidden, weight, cap=None):
    z = hidden.double() @ weight.double().t()
    return z if cap is None else cap * torch.tanh(z / cap)


@pytest.mark.parametrize("m,v,k,grid", [
    (1030, 33000, 64, 8),      # a few ties per row; an incomplete last tile and row tile
    (1030, 33000, 1, 8),
    (2049, 16640, 32, 2),      # hundreds of ties at the top: the scan
    (300, 131072, 256, 64),    # as many list entries as the path takes
])
def test_exact_on_representable_logits(gpu_device, m, v, k, grid):
    """Multiples of 1/grid with few bits: every sum is exact in float32 in any order."""
    print("[case]", m, v, k, grid, flush=True)
    gen = torch.Generator().manual_seed(v + k)
    h = 64
    hidden = (torch.randint(-grid, grid + 1, (m, h), generator=gen) / grid).bfloat16().to(gpu_device)
    weight = (torch.randint(-grid, grid + 1, (v, h), generator=gen) / grid).bfloat16().to(gpu_device)
    weight[: v // 64] *= 1.5   # the likely words sit together
    hidden[5] = 0.0                                        # all logits tie at 0
    labels = torch.randint(0, v, (m,), generator=gen).to(gpu_device)
    _, _, values, ids, _ = run(hidden, weight, labels, k)
    z = exact(hidden, weight)
    want_values, order = torch.sort(z, dim=1, descending=True, stable=True)
    assert torch.equal(ids, order[:, :k])
    assert torch.equal(values.double(), want_values[:, :k])


@pytest.mark.parametrize("cap", [None, 20.0])
def test_rows_that_need_another_way(gpu_device, cap):
    """Labels far below the row's maximum (the second try), so far above the other words that
    their entries underflow (the scan), rows of zeros, and ordinary rows, in one call; its
    gradient against float64: entries are rounded to bf16 once (1.66e-3 root mean square) and
    the result once more, so 2.35e-3 and less in the 2-norm."""
    m, h, v, k = 520, 256, 65000, 16
    gen = torch.Generator().manual_seed(3)
    weight = (torch.randn(v, h, generator=gen) * 0.05).bfloat16().to(gpu_device)
    labels = torch.randint(0, v, (m,), generator=gen).to(gpu_device)
    wy = weight[labels].float()
    hidden = torch.randn(m, h, generator=gen).to(gpu_device) * 2
    boost = torch.full((m, 1), 6.0, device=gpu_device)
    boost[::5] = -60.0
    if cap is None:
        boost[1::5] = 150.0
    hidden = (hidden + wy * (boost / wy.pow(2).sum(1, keepdim=True))).bfloat16()
    hidden[2] = 0.0
    up = torch.rand(3, m, generator=gen).to(gpu_device)
    loss, prob, values, ids, grad = run(hidden, weight, labels, k, cap, up)
    x = hidden.double().requires_grad_()
    z = exact(x, weight, cap)
    lse = torch.logsumexp(z, 1)
    want = lse - z.gather(1, labels[:, None])[:, 0]
    top = z.gather(1, ids)
    (want * up[0] + (-want).exp() * up[1] + top.mean(1) * up[2]).sum().backward()
    # lse and the label's logit are rounded at their own size (2^-24 each, and as much for
    # the sums behind them), and the loss is their difference
    assert bool(((loss.double() - want).abs() <= 1e-5 * want.abs() + 2.0 ** -22 * (1 + lse.abs())).all())
    assert torch.allclose(prob.double(), (-want).exp(), rtol=1e-4, atol=1e-9)   # 2^-22 * 150 and rounding
    assert torch.allclose(values.double(), top, rtol=1e-5, atol=1e-5)
    assert bool((values[:, 1:] <= values[:, :-1]).all())
    kth = z.topk(k, 1)[0][:, -1:]
    assert bool((top >= kth - 1e-4).all())                 # nothing larger was left out
    assert bool((ids.sort(1)[0].diff(dim=1) > 0).all())    # no word twice
    assert torch.equal(ids[2], torch.arange(k, device=gpu_device))
    error = float((grad.double() - x.grad).norm() / x.grad.norm())
    print("[case] gradient", error, flush=True)
    assert error < 2.35e-3
