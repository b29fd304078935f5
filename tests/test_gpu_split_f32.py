"""Float32 cross entropies on the bf16 matrix units (operands in three planes), where the
planes, the vocabulary chunks and panels, and the K passes have their edges.

Bound: an entry is a sum over K values taken 32 at a time, each step rounded in float32
(2^-24 relative to the running sum), plus the rounding of the logit (itself such a sum over
the hidden size), of the exponential (2 ulp) and of the result: 2-norm error below
2^-24 (8 + 2 sqrt(K / 32)) with K the longest of the three sums."""

import math

import pytest
import torch

from turbo_dllm_amd import _lib, options
from turbo_dllm_amd import chunked_linear_ce_native as native
from turbo_dllm_amd.tiled_linear_cross_entropy import tiled_linear_cross_entropy


def bound(*sums):
    return 2.0 ** -24 * (8 + 2 * math.sqrt(max(sums) / 32))


def operands(dev, m, h, v, seed, ignored=0.0):
    gen = torch.Generator().manual_seed(seed)
    weight = torch.randn(v, h, generator=gen) * 0.03
    labels = torch.randint(0, v - 1, (m,), generator=gen)
    hidden = torch.randn(m, h, generator=gen) + weight[labels] * (6.0 / (0.03 ** 2 * h))
    labels[torch.rand(m, generator=gen) < ignored] = -100
    return hidden.to(dev), weight.to(dev), labels.to(dev)


def exact(hidden, weight, labels, upstream, bias=None, softcap=0.0, exclude=-1):
    x, w = (t.double().requires_grad_() for t in (hidden, weight))
    z = x @ w.t()
    b = None
    if bias is not None:
        b = bias.double().requires_grad_()
        z = z + b
    if softcap:
        z = softcap * torch.tanh(z / softcap)
    if exclude >= 0:
        z = z.index_fill(1, torch.tensor([exclude], device=z.device), float("-inf"))
    losses = torch.nn.functional.cross_entropy(z, labels, reduction="none", ignore_index=-100)
    (losses * upstream).sum().backward()
    return losses.detach(), x.grad, w.grad, None if b is None else b.grad


def off(got, want):
    return float((got.double() - want).norm() / want.norm())


# rows around one and two 64-row K slabs past a tile, vocabularies with an incomplete slab,
# tile or neither, hidden sizes with an incomplete plane slab
CASES = [
    dict(m=385, h=512, v=16641),
    dict(m=513, h=516, v=16384, bias=True),
    dict(m=640, h=1024, v=12003, softcap=20.0, exclude=12002),
    dict(m=1030, h=580, v=8190, bias=True, softcap=15.0, ignored=0.3),
    dict(m=2049, h=768, v=4097, exclude=0, panel=24 << 20),
]


@pytest.mark.gpu
@pytest.mark.parametrize("mode", ["sync", "device", "none"])
@pytest.mark.parametrize("case", CASES, ids=lambda c: f"{c['m']}x{c['h']}x{c['v']}")
def test_planes_against_float64(gpu_device, case, mode):
    m, h, v = case["m"], case["h"], case["v"]
    print("[case]", case, mode, flush=True)
    hidden, weight, labels = operands(gpu_device, m, h, v, m, case.get("ignored", 0.0))
    gen = torch.Generator().manual_seed(1)
    upstream = (torch.rand(m, generator=gen) + 0.5).to(gpu_device)
    bias = (torch.randn(v, generator=gen) * 0.1).to(gpu_device) if case.get("bias") else None
    cap, exclude = case.get("softcap", 0.0), case.get("exclude", -1)
    want = exact(hidden, weight, labels, upstream, bias, cap, exclude)
    leaves = [t.clone().requires_grad_() for t in (hidden, weight)]
    b = None if bias is None else bias.clone().requires_grad_()
    with options.panel_budget(case.get("panel", 0)):
        losses = tiled_linear_cross_entropy(
            *leaves, labels, bias=b, reduction="none", logit_softcap=cap or None,
            exclude_index=exclude if exclude >= 0 else None, compaction=mode)
        (losses * upstream).sum().backward()
    got = (losses.detach(), leaves[0].grad, leaves[1].grad, None if b is None else b.grad)
    for g, w, name in zip(got, want, ("loss", "grad_hidden", "grad_weight", "grad_bias")):
        if w is not None:
            assert off(g, w) < bound(m, h, v), name


@pytest.mark.gpu
@pytest.mark.parametrize("reduction", ["mean", "sum"])
def test_one_and_several_vocabulary_chunks(gpu_device, reduction):
    """A head whose planes exceed their bound is taken in chunks, forward and backward."""
    m, h, v = 400, 8192, 22001
    assert v * h * 6 > 1 << 30
    hidden, weight, labels = operands(gpu_device, m, h, v, 5)
    scale = torch.full((m,), 1.0 / m if reduction == "mean" else 1.0, device=gpu_device)
    want = exact(hidden, weight, labels, scale, exclude=v - 1)
    for frozen in (False, True):
        x, w = hidden.clone().requires_grad_(), weight.clone().requires_grad_(not frozen)
        loss = tiled_linear_cross_entropy(x, w, labels, reduction=reduction, exclude_index=v - 1)
        loss.backward()
        assert off(loss.detach(), (want[0] * scale).sum()) < bound(m, h, v)
        assert off(x.grad, want[1]) < bound(m, h, v)
        assert frozen or off(w.grad, want[2]) < bound(m, h, v)


@pytest.mark.gpu
def test_vocabulary_shards_in_planes(gpu_device):
    """Two shards, both in planes, combine to the loss and gradients of the whole head."""
    m, h, v = 520, 512, 26000
    hidden, weight, labels = operands(gpu_device, m, h, v, 9)
    want = exact(hidden, weight, labels, torch.ones(m, device=gpu_device))
    parts = [(0, 13001), (13001, v)]
    stats = [native.vocab_parallel_forward_local(
        hidden, weight[a:b], None, labels, vocab_start=a, ignore_index=-100, exclude_index=-1,
        logit_softcap=0.0) for a, b in parts]
    top = torch.stack([s[0] for s in stats]).amax(0)
    total = sum(s[1] * torch.exp(s[0] - top) for s in stats)
    target = sum(s[2] for s in stats)
    lse = top + total.log()
    assert off(lse - target, want[0]) < bound(m, h, v)


@pytest.mark.gpu
def test_values_at_the_ends_of_float32(gpu_device):
    """Rows of zeros, of tiny and of huge numbers: the planes neither overflow nor turn
    what is finite into NaN."""
    m, h, v = 512, 512, 16384
    hidden, weight, labels = operands(gpu_device, m, h, v, 3)
    hidden[0] = 0.0
    hidden[1] *= 1e-30
    weight[7] = 0.0
    weight[8] = 0.0
    weight[8, 0] = torch.finfo(torch.float32).max
    hidden[:, 0] = 0.0
    losses = tiled_linear_cross_entropy(hidden, weight, labels, reduction="none")
    want = torch.nn.functional.cross_entropy(hidden.double() @ weight.double().t(), labels,
                                             reduction="none")
    assert torch.isfinite(losses).all()
    assert off(losses, want) < bound(h, v)


def test_scratch_of_the_planes_is_bounded():
    lib = _lib.library()
    f32 = _lib.DTYPE_F32
    mib = 1 << 20
    # taken: more scratch than the partials; not taken (rows, tiles, hidden size): partials
    assert lib.tlce_forward_workspace_bytes(1024, 1024, 32000, f32) > 190 * mib
    for m, h, v in ((384, 1024, 32000), (1024, 508, 32000), (1024, 1022, 32000),
                    (1024, 1024, 7936), (65536, 1024, 2047)):
        assert lib.tlce_forward_workspace_bytes(m, h, v, f32) <= 4 * mib
    # the planes of a large head: 1 GiB at a time, beside those of the hidden rows
    hidden = 2048 * 4096 * 6
    assert lib.tlce_forward_workspace_bytes(2048, 4096, 262144, f32) < 1024 * mib + hidden + 4 * mib
    backward = lib.tlce_backward_workspace_bytes(2048, 4096, 262144, f32, 1, 0, 0)
    assert backward < 2 * 1024 * mib + hidden + 64 * 2048 * 4096 * 4


def launches_of(call):
    """Launches per kernel class of what `call` runs (forward only: this thread)."""
    with _lib.kernel_profile() as prof:
        result = call()
        torch.cuda.synchronize()
    return result, prof


@pytest.mark.gpu
@pytest.mark.parametrize("mode", ["sync", "device", "none"])
@pytest.mark.parametrize("case", [
    dict(m=129, h=512, v=24449, reduction="mean"),
    dict(m=1500, h=580, v=8190, reduction="sum", softcap=15.0, exclude=8189, ignored=0.3),
    dict(m=1030, h=580, v=8190, reduction="none", frozen=True),
    # blocks of 256 rows, the last of one row
    dict(m=1025, h=640, v=8191, reduction="mean", panel=14 << 20),
    # losses beyond the first try's window in some rows
    dict(m=520, h=512, v=16384, reduction="sum", far=True),
], ids=lambda c: f"{c['m']}x{c['h']}x{c['v']}-{c['reduction']}")
def test_gradients_left_by_the_forward(gpu_device, case, mode):
    m, h, v = case["m"], case["h"], case["v"]
    print("[case]", case, mode, flush=True)
    hidden, weight, labels = operands(gpu_device, m, h, v, m, case.get("ignored", 0.0))
    if case.get("far"):
        hidden[::7] *= 20.0
        labels[::7] = (labels[::7] + 1) % v
    valid = labels != -100
    cap, exclude = case.get("softcap", 0.0), case.get("exclude", -1)
    upstream = torch.ones(m, device=gpu_device)
    if case["reduction"] == "mean":
        upstream /= valid.sum()
    if case["reduction"] == "none":
        upstream = (torch.rand(m, generator=torch.Generator().manual_seed(2)) + 0.5).to(gpu_device)
    want = exact(hidden, weight, labels, upstream, None, cap, exclude)
    x = hidden.clone().requires_grad_()
    w = weight.clone().requires_grad_(not case.get("frozen", False))
    with options.panel_budget(case.get("panel", 0)):
        loss, prof = launches_of(lambda: tiled_linear_cross_entropy(
            x, w, labels, reduction=case["reduction"], logit_softcap=cap or None,
            exclude_index=exclude if exclude >= 0 else None, compaction=mode))
        assert prof.launches["exp_logits_panel"] > 0
        for again in (False, True):   # a second backward over one graph
            x.grad = w.grad = None
            (loss * upstream).sum().backward(retain_graph=True) \
                if case["reduction"] == "none" else loss.backward(retain_graph=True)
            # (an entry is formed from two sums over the vocabulary, a hidden one and a factor)
            assert off(x.grad, want[1]) < 2 * bound(m, h, v)
            assert case.get("frozen") or off(w.grad, want[2]) < 2 * bound(m, h, v)
    total = want[0] if case["reduction"] == "none" else (want[0] * upstream).sum()
    assert off(loss.detach(), total) < bound(m, h, v)


@pytest.mark.gpu
def test_masked_token_loss_in_planes(gpu_device):
    """Token weights and the output multiplier, which enter the row factors."""
    from turbo_dllm_amd.loss import masked_token_loss
    m, h, v = 700, 512, 16001
    hidden, weight, labels = operands(gpu_device, m, h, v, 4, 0.1)
    weights = (torch.rand(m, generator=torch.Generator().manual_seed(6)) + 0.5).to(gpu_device)
    head = torch.nn.Linear(h, v, bias=False, device=gpu_device)
    head.weight = torch.nn.Parameter(weight)
    x = hidden.clone().requires_grad_()
    loss = masked_token_loss(x, labels, weights, head, valid_token_count=100.0,
                             mask_token_id=v - 1, output_multiplier=0.5)
    loss.backward()
    want = exact(hidden * 0.5, weight, labels, weights / 100.0, exclude=v - 1)
    assert off(loss.detach(), (want[0] * weights / 100.0).sum()) < bound(m, h, v)
    assert off(x.grad, 0.5 * want[1]) < 2 * bound(m, h, v)
    assert off(head.weight.grad, want[2]) < 2 * bound(m, h, v)


def test_which_float32_calls_leave_their_gradients_in_the_forward():
    taken = _lib.library().tlce_f32_gradients_in_forward_supported
    assert taken(1024, 1024, 32000) and taken(385, 512, 16641)
    assert taken(129, 1024, 32000) and not taken(128, 1024, 32000)      # rows
    assert not taken(1024, 1024, 5888)            # tiles
    assert not taken(2048, 4096, 151936)          # a head of more than 1 GiB of planes
    assert not taken(1024, 1022, 32000)           # hidden size
    size = _lib.library().tlce_forward_with_gradients_f32_workspace_bytes
    assert size(128, 1024, 32000, 1, 0) == -1
    assert 0 < size(65536, 1024, 32000, 1, 0) < (5 << 29) + (2 << 30)
