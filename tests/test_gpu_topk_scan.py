"""The scan of the float32 logits panels of the CE with exact top-k at the edges of its
16384-column chunks and of its ways of finding a first threshold (k up to 32 by waves, above
by all threads).  Inputs are small multiples of 1/8, so every logit is exact in float32 in
any order of summation and has exact ties: values and ids must be the oracle's, ties going
to the smaller id.  Loss within 1e-5 and the gradient within 1e-2 relative max-norm of the
float64 oracle (softmax entries rounded to bf16 once, twice where a row's maximum grew:
2 * 2^-9 relative at most, plus one rounding of the result)."""

import pytest
import torch

import linear_ce_oracle as oracle
from turbo_dllm_amd import chunked_linear_ce_native as native
from turbo_dllm_amd import options
from turbo_dllm_amd.dflash_linear_topk import frozen_linear_ce_topk

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m,v,k,panel_tiles,softcap", [
    (1, 64, 1, 0, None),             # most threads hold no column
    (3, 64, 64, 0, None),            # k is the vocabulary
    (5, 1500, 20, 0, None),          # six of eight waves are empty; fewer columns than threads * 4
    (257, 16384, 32, 0, None),       # one whole chunk, a row past a tile
    (130, 16385, 33, 0, 30.0),       # one column in the second chunk
    (64, 33000, 16, 0, None),        # three chunks, the vocabulary ends inside a tile
    (70, 50000, 64, 80, None),       # panels of 20480 columns: chunks of 16384 and 4096
    (40, 40960, 16, 64, 30.0),       # panels of one chunk each
])
def test_scan_edges(gpu_device, m, v, k, panel_tiles, softcap):
    print("[case]", m, v, k, panel_tiles, softcap, flush=True)
    gen = torch.Generator().manual_seed(m + v)
    hidden = (torch.randint(-8, 9, (m, 64), generator=gen) / 8).bfloat16()
    weight = (torch.randint(-4, 5, (v, 64), generator=gen) / 8).bfloat16()
    # maxima that grow towards the end of the vocabulary
    weight[-max(1, v // 8):] *= 2
    labels = torch.randint(0, v, (m,), generator=gen)
    rows = -(-m // 256) * 256
    x = hidden.to(gpu_device).requires_grad_(True)
    up = torch.rand(3, m, generator=gen)
    with options.panel_budget(panel_tiles * 256 * rows * 4):
        loss, prob, values, ids = frozen_linear_ce_topk(
            x, weight.to(gpu_device), labels.to(gpu_device), top_k=k, logit_softcap=softcap)
        g = up.to(gpu_device)
        (loss * g[0] + prob * g[1] + values.mean(1) * g[2]).sum().backward()
    torch.cuda.synchronize()
    raw = hidden.double() @ weight.double().t()
    # (capped logits keep the order of the raw ones; ties of capped float32 values are
    # not ties of the oracle's)
    order = torch.argsort(raw, dim=1, descending=True, stable=True)[:, :k]
    z = raw if softcap is None else softcap * torch.tanh(raw / softcap)
    if softcap is None:
        assert torch.equal(ids.cpu(), order)
        assert torch.equal(values.detach().cpu().double(), raw.gather(1, order))
    else:
        assert torch.allclose(values.detach().cpu().double(), z.gather(1, order), rtol=1e-5, atol=1e-5)
    want = torch.logsumexp(z, 1) - z.gather(1, labels[:, None])[:, 0]
    assert torch.allclose(loss.detach().cpu().double(), want, rtol=1e-5, atol=1e-5)
    grad = oracle.dense_ce_topk_grad(hidden, weight, labels, ids.cpu(), up[0], up[1],
                                     up[2][:, None].expand(m, k) / k, logit_softcap=softcap)
    error = oracle.relative_max_error(x.grad, grad)
    print("[case] gradient error", error, flush=True)
    assert error <= 1e-2


def test_entries_of_one_logits_panel_are_rounded_once(gpu_device):
    """Three chunks of the scan in one float32 logits panel, the row maximum in the last of
    them: the entries of the gradient panel are exp(logit - maximum of the panel) rounded to
    bf16 once, so d lse / d hidden is as far from float64 as that one rounding makes it (5 %
    for hardware exponentials that round the other way; entries rounded in the chunk they
    are scanned in, and again for the final maximum, are about 1.4 times as far)."""
    m, h, v = 64, 64, 49152
    gen = torch.Generator().manual_seed(7)
    hidden = (torch.randint(-8, 9, (m, h), generator=gen) / 8).bfloat16().to(gpu_device)
    weight = (torch.randint(-2, 3, (v, h), generator=gen) / 8).bfloat16().to(gpu_device)
    weight[:, 0] += (torch.arange(v, device=gpu_device) // 16384) * 0.5   # later words are likelier
    hidden[:, 0] = 1.0
    labels = torch.randint(0, v, (m,), generator=gen).to(gpu_device)
    unit = native.dflash_ce_topk_forward_with_gradient(
        hidden, weight, labels, top_k=4, output_multiplier=1.0, logit_softcap=0.0)[5]
    z = hidden.double() @ weight.double().t()
    maxima = [z[:, c:c + 16384].amax(1) for c in range(0, v, 16384)]
    assert float((maxima[0] < maxima[2]).double().mean()) > 0.5
    e = (z - z.amax(1, keepdim=True)).exp()
    exact = (e @ weight.double()) / e.sum(1, keepdim=True)
    once = (e.bfloat16().double() @ weight.double()) / e.sum(1, keepdim=True)
    error, bound = float((unit.double() - exact).norm()), float((once - exact).norm())
    print("[case] error", error / float(exact.norm()), "one rounding", bound / float(exact.norm()), flush=True)
    assert error <= 1.05 * bound
