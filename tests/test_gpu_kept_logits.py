"""Logits that a forward keeps for its backward (``kept_logits_buffer``): the gradients of a
backward that recomputes them, bit for bit, over every kind of operand the kept tiles take:
edges of tiles, an excluded word, soft caps, ignored rows, heads stored [H, V], hidden sizes
that are no multiple of 64, and buffers that hold a part of the vocabulary, which may end inside
a panel of the backward."""

import pytest
import torch
import torch.utils.checkpoint

from turbo_dllm_amd import _lib, options
from turbo_dllm_amd import chunked_linear_ce_native as native
from turbo_dllm_amd.loss import masked_token_loss, native_token_cross_entropy
from turbo_dllm_amd.tiled_linear_cross_entropy import tiled_linear_cross_entropy

pytestmark = pytest.mark.gpu

TILE_BYTES = 256 * 256 * 4


def operands(dev, m, h, v, dtype=torch.bfloat16, ignored=0.0):
    print("[case]", m, h, v, dtype, ignored, flush=True)
    gen = torch.Generator(device=dev).manual_seed(m + 3 * h + v)
    hidden = torch.randn(m, h, generator=gen, device=dev).to(dtype)
    weight = (torch.randn(v, h, generator=gen, device=dev) * 0.03).to(dtype)
    labels = torch.randint(0, v - 1, (m,), generator=gen, device=dev)
    labels[torch.rand(m, generator=gen, device=dev) < ignored] = -100
    up = torch.rand(m, generator=gen, device=dev) / m
    return hidden, weight, labels, up


def step(hidden, weight, labels, up, reduction, trainable=True, **keywords):
    x = hidden.detach().clone().requires_grad_()
    w = weight.detach().clone().requires_grad_(trainable)
    loss = tiled_linear_cross_entropy(x, w, labels, reduction=reduction, dtype=x.dtype, **keywords)
    (loss * up).sum().backward() if reduction == "none" else loss.backward()
    return [loss.detach(), x.grad] + ([w.grad] if trainable else [])


class Spy:
    """Counts the bytes the calls inside the block keep."""

    def __init__(self, monkeypatch):
        self.kept = []
        inner = native.kept_logits_buffer

        def spy(*args):
            buffer = inner(*args)
            self.kept.append(0 if buffer is None else buffer.numel())
            return buffer

        monkeypatch.setattr(native, "kept_logits_buffer", spy)


def same_as_recomputed(spy, call):
    del spy.kept[:]
    got = call()
    assert len(spy.kept) == 1 and spy.kept[0] > 0
    with options.gradient_mode("recompute"):
        want = call()
    assert spy.kept[1:] == [0]
    for a, b in zip(got, want):
        assert torch.equal(a, b)
    return spy.kept[0]


@pytest.mark.parametrize("m,h,v,dtype,reduction,keywords", [
    (600, 1024, 3001, torch.bfloat16, "mean", {}),
    (257, 1088, 515, torch.bfloat16, "sum", {"exclude_index": 514}),
    (256, 1024, 4096, torch.float16, "mean", {}),
    (1, 1024, 257, torch.float16, "none", {"logit_softcap": 30.0}),
    (600, 1032, 9001, torch.bfloat16, "mean", {"logit_softcap": 20.0}),     # column tail
    (520, 2040, 9000, torch.float16, "none", {"exclude_index": 255}),
    (513, 1024, 2049, torch.bfloat16, "none", {"logit_softcap": 30.0, "exclude_index": 2048}),
])
@pytest.mark.parametrize("ignored", [0.0, 0.4])
def test_kept_logits_give_the_recomputed_gradients(gpu_device, monkeypatch, m, h, v, dtype,
                                                   reduction, keywords, ignored):
    hidden, weight, labels, up = operands(gpu_device, m, h, v, dtype, ignored if m > 1 else 0.0)
    spy = Spy(monkeypatch)
    size = same_as_recomputed(spy, lambda: step(hidden, weight, labels, up, reduction, **keywords))
    assert size % TILE_BYTES == 0
    frozen = v % 64 != 0 or dtype == torch.float16      # (whole slabs under a frozen head: no)
    if frozen:
        same_as_recomputed(
            spy, lambda: step(hidden, weight, labels, up, reduction, trainable=False, **keywords))


@pytest.mark.parametrize("v,dtype", [(4096, torch.float16), (4032, torch.bfloat16)])
def test_a_head_stored_dim_first(gpu_device, monkeypatch, v, dtype):
    hidden, weight, labels, up = operands(gpu_device, 700, 1024, v, dtype, 0.3)
    dim_first = weight.t().contiguous()
    same_as_recomputed(Spy(monkeypatch), lambda: step(hidden, dim_first, labels, up, "mean",
                                                      weight_layout="dim_first"))


@pytest.mark.parametrize("tiles", [1, 3, 7, 11, 12])
@pytest.mark.parametrize("panel_tiles", [2, 5])
def test_a_buffer_for_part_of_the_vocabulary(gpu_device, monkeypatch, tiles, panel_tiles):
    """12 vocabulary tiles in panels of two or five, the first `tiles` kept."""
    m, h, v = 600, 1024, 3001
    hidden, weight, labels, up = operands(gpu_device, m, h, v)
    budget = native._lib.library().tlce_kept_logits_bytes(
        m, h, v, _lib.DTYPE_BF16, 0, tiles * 3 * TILE_BYTES + 1000)
    assert budget == tiles * 3 * TILE_BYTES
    kept = torch.empty(budget, dtype=torch.uint8, device=gpu_device)
    arguments = dict(ignore_index=-100, exclude_index=-1, logit_softcap=0.0)
    results = []
    for buffer in (kept, None):
        losses, lse, count, _ = native.masked_loss_forward(
            hidden, weight, None, labels, None, want_sum=False, kept=buffer, **arguments)
        with native.panel_budget(768 * 256 * 2 * panel_tiles):
            results.append([losses, lse, *native.masked_loss_backward(
                hidden, weight, None, labels, None, lse, count, up, reduction="none",
                kept=buffer, **arguments)[:2]])
    for a, b in zip(*results):
        assert torch.equal(a, b)


def test_the_losses_built_on_it(gpu_device, monkeypatch):
    hidden, weight, labels, up = operands(gpu_device, 700, 1024, 3003, ignored=0.3)
    spy = Spy(monkeypatch)
    head = torch.nn.Linear(1024, 3003, bias=False, device=gpu_device, dtype=torch.bfloat16)
    head.weight = torch.nn.Parameter(weight)

    def masked():
        x = hidden.detach().clone().requires_grad_()
        head.weight.grad = None
        loss = masked_token_loss(x, labels, up, head, valid_token_count=500.0, mask_token_id=3002,
                                 output_multiplier=0.5, logit_softcap=30.0)
        loss.backward()
        return [loss.detach(), x.grad, head.weight.grad]

    def tokens():
        x = hidden.detach().clone().requires_grad_()
        head.weight.grad = None
        losses = native_token_cross_entropy(x, labels.clamp(min=0), head, output_multiplier=0.5)
        (losses * up).sum().backward()
        return [losses.detach(), x.grad, head.weight.grad]

    same_as_recomputed(spy, masked)
    same_as_recomputed(spy, tokens)


def test_what_keeps_nothing(gpu_device, monkeypatch):
    spy = Spy(monkeypatch)
    for m, h, v, dtype in ((600, 960, 3001, torch.bfloat16), (600, 1028, 3001, torch.float32)):
        hidden, weight, labels, up = operands(gpu_device, m, h, v, dtype)
        step(hidden, weight, labels, up, "none")
    assert spy.kept and not any(spy.kept)
    hidden, weight, labels, up = operands(gpu_device, 600, 1024, 3001)
    bias = torch.zeros(3001, dtype=torch.bfloat16, device=gpu_device)
    step(hidden, weight, labels, up, "mean", bias=bias)
    with torch.no_grad():
        tiled_linear_cross_entropy(hidden, weight, labels, dtype=torch.bfloat16)
    with native.panel_budget(TILE_BYTES):
        step(hidden, weight, labels, up, "mean")
    step(hidden, weight, labels, up, "mean", compaction="device")
    assert not any(spy.kept)
    with pytest.raises(RuntimeError):      # a buffer these operands cannot have
        native.masked_loss_forward(
            hidden.float(), weight.float(), None, labels, None, ignore_index=-100, exclude_index=-1,
            logit_softcap=0.0, kept=torch.empty(1 << 20, dtype=torch.uint8, device=gpu_device))


def test_a_backward_without_memory_beside_the_logits(gpu_device, monkeypatch):
    """It recomputes them in the place they are given back from: the same gradients."""
    hidden, weight, labels, up = operands(gpu_device, 600, 1024, 3001, ignored=0.4)
    inner, refused = native.masked_loss_backward, []

    def without_memory(*args, kept=None, **keywords):
        if kept is not None:
            refused.append(kept)
            raise torch.OutOfMemoryError("no room")
        return inner(*args, kept=kept, **keywords)

    want = step(hidden, weight, labels, up, "none")
    monkeypatch.setattr(native, "masked_loss_backward", without_memory)
    got = step(hidden, weight, labels, up, "none")
    assert len(refused) == 1 and refused[0].untyped_storage().size() == 0
    for a, b in zip(got, want):
        assert torch.equal(a, b)


@pytest.mark.parametrize("loss", ["ce", "tokens", "masked"])
def test_checkpointing_while_free_memory_changes(gpu_device, monkeypatch, loss):
    """Non-reentrant checkpointing compares what the forward and its repetition save: logits for
    which there is room in one of them only must not be among it."""
    hidden, weight, labels, up = operands(gpu_device, 600, 1024, 3001)
    head = torch.nn.Linear(1024, 3001, bias=False, device="meta")
    left = [1 << 40]
    monkeypatch.setattr(torch.cuda, "mem_get_info", lambda device: (left[0], 1 << 40))
    monkeypatch.setattr(native, "_memory_cached", lambda device: 0)
    monkeypatch.setattr(native, "_KEEP_UNASKED_BYTES", 0)

    def gradients(wrap):
        x = hidden.clone().requires_grad_()
        head.weight = w = torch.nn.Parameter(weight.clone())

        def forward(x):
            if loss == "ce":
                return (tiled_linear_cross_entropy(x, w, labels, reduction="none",
                                                   dtype=x.dtype) * up).sum()
            if loss == "tokens":
                return (native_token_cross_entropy(x, labels, head) * up).sum()
            return masked_token_loss(x, labels, up, head, valid_token_count=600.0)

        left[0] = 1 << 40
        result = wrap(forward, x)
        left[0] = 0
        result.backward()
        return [result.detach(), x.grad, w.grad]

    want = gradients(lambda forward, x: forward(x))
    got = gradients(lambda forward, x: torch.utils.checkpoint.checkpoint(
        forward, x, use_reentrant=False))
    for a, b in zip(got, want):
        assert torch.equal(a, b)
