"""Small calls whose count of rows with a loss stays on the device in the default compaction
(``native.count_stays_on_device``): no host synchronisation, and the results of a call that
compacts nothing, for no row with a loss up to all of them, around tiles and 64-row slabs.  The
same with the count read back, as larger calls have it."""

import pytest
import torch

from turbo_dllm_amd import chunked_linear_ce_native as native, options
from turbo_dllm_amd.loss import masked_token_loss
from turbo_dllm_amd.tiled_linear_cross_entropy import tiled_linear_cross_entropy

pytestmark = pytest.mark.gpu

N = 700
SHAPES = [(256, 1088, torch.bfloat16),      # gradients in the forward
          (1024, 1091, torch.bfloat16),     # kept logits: odd vocabulary,
          (1024, 1088, torch.float16),      # float16,
          (1032, 3008, torch.bfloat16)]     # column tail


@pytest.fixture(scope="module", params=SHAPES, ids=str)
def operands(gpu_device, request):
    h, v, dtype = request.param
    gen = torch.Generator(device=gpu_device).manual_seed(2)
    hidden = torch.randn(N, h, generator=gen, device=gpu_device).to(dtype)
    weight = (torch.randn(v, h, generator=gen, device=gpu_device) * 0.05).to(dtype)
    labels = torch.randint(0, v - 1, (N,), generator=gen, device=gpu_device)
    order = torch.rand(N, generator=gen, device=gpu_device).argsort()
    up = torch.rand(N, generator=gen, device=gpu_device)
    return hidden, weight, labels, order, up


def read_back(monkeypatch):
    for rule in ("count_stays_on_device", "kept_count_stays_on_device"):
        monkeypatch.setattr(native, rule, lambda *args: False)


def without_synchronisation(call):
    call()          # (allocations and first launches)
    torch.cuda.synchronize()
    torch.cuda.set_sync_debug_mode("error")
    try:
        return call()
    finally:
        torch.cuda.set_sync_debug_mode("default")


def close(got, want):
    for a, b in zip(got, want):
        assert torch.equal(a.isnan(), b.isnan())
        a, b = a.nan_to_num().double(), b.nan_to_num().double()
        # (the same float32 sums in another order, each rounded to bf16: one ulp of the largest
        # entry apart, 2^-7 of it with 8 significant bits)
        assert (a - b).abs().max() <= 2.0 ** -7 * a.abs().max() + 1e-12


@pytest.mark.parametrize("reduction", ["mean", "sum", "none"])
@pytest.mark.parametrize("trainable", [True, False])
@pytest.mark.parametrize("kept", [0, 1, 64, 65, 255, 256, 257, 384, 513, N - 1, N])
@pytest.mark.parametrize("counted", [False, True])
def test_cross_entropy(operands, monkeypatch, reduction, trainable, kept, counted):
    hidden, weight, labels, order, up = operands
    labels = labels.clone()
    labels[order[kept:]] = -100
    v = weight.shape[0]
    assert (native.count_stays_on_device(N, hidden, weight, None, False)
            or native.kept_count_stays_on_device(N, hidden, weight, None, trainable))

    def step(compaction):
        x = hidden.clone().requires_grad_()
        w = weight.clone().requires_grad_(trainable)
        loss = tiled_linear_cross_entropy(x, w, labels, reduction=reduction, dtype=x.dtype,
                                          exclude_index=v - 1, compaction=compaction)
        (loss * up if reduction == "none" else loss).sum().backward()
        return [loss.detach(), x.grad] + ([w.grad] if trainable else [])

    if counted:
        read_back(monkeypatch)
        got = step("sync")
    else:
        got = without_synchronisation(lambda: step("sync"))
    if kept == 0 and reduction == "mean":
        assert got[0].isnan()       # the mean over no row, as before
        return
    close(got, step("none"))


@pytest.mark.parametrize("kept", [0, 1, 257, N])
@pytest.mark.parametrize("counted", [False, True])
def test_masked_token_loss(operands, monkeypatch, kept, counted):
    hidden, weight, labels, order, up = operands
    labels = labels.clone()
    labels[order[kept:]] = -100
    v, h = weight.shape
    head = torch.nn.Linear(h, v, bias=False, device=hidden.device, dtype=hidden.dtype)

    def step(mode):
        x = hidden.clone().requires_grad_()
        head.weight = torch.nn.Parameter(weight.clone())
        with options.compaction_mode(mode):
            loss = masked_token_loss(x, labels, up, head, valid_token_count=300.0,
                                     mask_token_id=v - 1, exclude_mask_token=True,
                                     output_multiplier=0.5, logit_softcap=20.0)
            loss.backward()
        return [loss.detach(), x.grad, head.weight.grad]

    want = step("none")
    if counted:
        read_back(monkeypatch)
        close(step("sync"), want)
    else:
        close(without_synchronisation(lambda: step("sync")), want)


def test_captured_with_any_count(operands):
    """No synchronisation, so such a call can be captured in the default compaction: replayed with
    other counts and eager steps in between, the bits of the eager step (which keeps logits where
    the captured one recomputes them)."""
    hidden, weight, labels, order, _ = operands
    x = hidden.clone().requires_grad_()
    w = weight.clone().requires_grad_()
    y = labels.clone()

    def step():
        loss = tiled_linear_cross_entropy(x, w, y, reduction="sum", dtype=x.dtype)
        return [loss.detach(), *torch.autograd.grad(loss, (x, w))]

    side = torch.cuda.Stream()
    with torch.cuda.stream(side):
        step()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        outputs = step()
    for kept in (N, 3, 257, 0, 600):
        y.copy_(labels)
        y[order[kept:]] = -100
        graph.replay()
        torch.cuda.synchronize()
        got = [t.clone() for t in outputs]
        for a, b in zip(got, step()):
            assert torch.equal(a, b), kept


@pytest.mark.parametrize("h,v,trainable", [
    (256, 16384, True), (320, 9024, True),       # gradients in the forward,
    (3840, 16384, True),                         # 8 splits of 2 tiles, 5 of 3,
    (1024, 9001, True), (1032, 20001, False)])   # kept logits
@pytest.mark.parametrize("kept", [1, 64, 65, 256, 300, 513, N - 1])
def test_the_bits_of_a_counted_call(gpu_device, monkeypatch, h, v, trainable, kept):
    """Few tiles over many words: as many K splits, and so the same sums, as with a known count."""
    print("[case]", h, v, trainable, kept, flush=True)
    gen = torch.Generator(device=gpu_device).manual_seed(h + kept)
    hidden = torch.randn(N, h, generator=gen, device=gpu_device).bfloat16()
    weight = (torch.randn(v, h, generator=gen, device=gpu_device) * 0.05).bfloat16()
    labels = torch.randint(0, v, (N,), generator=gen, device=gpu_device)
    labels[torch.rand(N, generator=gen, device=gpu_device).argsort()[kept:]] = -100

    def step():
        x = hidden.clone().requires_grad_()
        w = weight.clone().requires_grad_(trainable)
        loss = tiled_linear_cross_entropy(x, w, labels, dtype=x.dtype)
        loss.backward()
        return [loss.detach(), x.grad] + ([w.grad] if trainable else [])

    got = without_synchronisation(step)
    read_back(monkeypatch)
    for a, b in zip(got, step()):
        assert torch.equal(a, b)


def test_larger_calls_are_counted(gpu_device):
    for n, h, stays in ((4096, 1024, True), (4097, 1024, False), (4096, 960, False)):
        rows = torch.empty(n, h, dtype=torch.float16, device=gpu_device)
        head = torch.empty(32768, h, dtype=torch.float16, device=gpu_device)
        assert native.kept_count_stays_on_device(n, rows, head, None, True) == stays
    small = torch.empty(4096, 64, dtype=torch.bfloat16, device=gpu_device)
    for vocab, stays in ((32768, True), (32832, False)):
        head = torch.empty(vocab, 64, dtype=torch.bfloat16, device=gpu_device)
        assert native.count_stays_on_device(4096, small, head, None, False) == stays
    assert not native.count_stays_on_device(256, small[:256], head, None, False)
    with native.panel_budget(1 << 20):      # several blocks
        assert not native.count_stays_on_device(4096, small, head[:4096], None, False)
