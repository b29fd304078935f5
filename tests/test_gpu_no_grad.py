"""Without grad mode the losses form no gradients, whatever their operands require: one
contraction (KL: two), and the same numbers bit for bit as detached operands give."""

import pytest
import torch

from turbo_dllm_amd import _lib
from turbo_dllm_amd import chunked_linear_ce_native as native
from turbo_dllm_amd.dflash_kl import frozen_linear_kl
from turbo_dllm_amd.dflash_linear_topk import frozen_linear_ce_topk
from turbo_dllm_amd.loss import dflash_token_loss, masked_token_loss, native_token_cross_entropy
from turbo_dllm_amd.tiled_linear_cross_entropy import tiled_linear_cross_entropy

pytestmark = pytest.mark.gpu


def cross_entropy(reduction, dim_first=False):
    def call(x, w, y, up):
        return tiled_linear_cross_entropy(
            x, w.t() if dim_first else w, y, reduction=reduction, dtype=x.dtype,
            weight_layout="dim_first" if dim_first else "vocab_first")
    return call


def masked(x, w, y, up):
    head = torch.nn.Linear(w.shape[1], w.shape[0], bias=False, device="meta")
    head.weight = w
    return masked_token_loss(x, y, up, head, valid_token_count=float(len(y)),
                             exclude_mask_token=False)


def drafter(x, w, y, up):
    head = torch.nn.Linear(w.shape[1], w.shape[0], bias=False, device="meta")
    head.weight = w
    counts = torch.full((2,), 9.0, device=x.device)
    return dflash_token_loss(x.reshape(2, -1, x.shape[1]), y.reshape(2, -1),
                             (y != -100).reshape(2, -1), up.reshape(2, -1), head,
                             loss_kind="paper_ce", normalization_count=counts)


def tokens(x, w, y, up):
    head = torch.nn.Linear(w.shape[1], w.shape[0], bias=False, device="meta")
    head.weight = w
    return native_token_cross_entropy(x, y, head, output_multiplier=0.5)


def top_k(x, w, y, up):
    return torch.cat([t.flatten().double() for t in
                      frozen_linear_ce_topk(x, w.detach(), y.clamp(min=0), top_k=4)])


def kl(x, w, y, up):
    return frozen_linear_kl(x, w.detach(), x.detach(), w.detach() * 0.5)


CALLS = {"none": cross_entropy("none"), "mean": cross_entropy("mean"),
         "dim_first": cross_entropy("sum", dim_first=True), "masked": masked, "drafter": drafter,
         "tokens": tokens, "top_k": top_k, "kl": kl}
SIZES = [
    (200, 192, 1600, torch.bfloat16),       # rows of one tile
    (700, 256, 3008, torch.bfloat16),
    (3500, 1920, 32001, torch.bfloat16),    # no whole slabs
    (600, 512, 16400, torch.float32),       # in planes
    (700, 256, 3008, torch.float16),
]


@pytest.mark.parametrize("m,h,v,dtype,kind", [
    (*size, kind) for size in SIZES for kind in CALLS
    if size[3] != torch.float32 or kind != "top_k"])    # (which is plain torch there)
@pytest.mark.parametrize("inference", [False, True])
def test_no_gradients_are_formed(gpu_device, monkeypatch, m, h, v, dtype, kind, inference):
    print("[case]", m, h, v, dtype, kind, inference, flush=True)
    gen = torch.Generator().manual_seed(m)
    x = torch.randn(m, h, generator=gen).to(dtype).to(gpu_device)
    w = (torch.randn(v, h, generator=gen) * 0.03).to(dtype).to(gpu_device)
    y = torch.randint(0, v, (m,), generator=gen)
    y[torch.rand(m, generator=gen) < 0.3] = -100
    y = y.to(gpu_device)
    up = (torch.rand(m, generator=gen) + 0.5).to(gpu_device)
    call = CALLS[kind]

    def keep(*args):
        raise AssertionError("logits kept for no backward")

    monkeypatch.setattr(native, "kept_logits_buffer", keep)
    with torch.no_grad():
        want = call(x, torch.nn.Parameter(w, requires_grad=False), y, up)
    x = x.requires_grad_()
    with torch.inference_mode() if inference else torch.no_grad(), _lib.kernel_profile() as prof:
        got = call(x, torch.nn.Parameter(w), y, up)
    assert not got.requires_grad and torch.equal(got, want)
    for made in ("exp_logits_panel", "grad_logits_panel", "grad_hidden_gemm", "grad_weight_gemm"):
        # (that class counts the panels of the teacher and of float32 logits as well)
        if made != "grad_logits_panel" or kind not in ("kl", "top_k"):
            assert prof.launches[made] == 0, prof.launches
