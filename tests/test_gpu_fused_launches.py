"""The calls that join launches (the loss summed by the slab reduction, labels, counts and
clearing in one launch, one pass over rows in the backward) against the calls they replace:
gradients bit for bit; the loss is a sum of n float32 numbers in another order (n * 2^-24)."""

import pytest
import torch

from turbo_dllm_amd import chunked_linear_ce_native as native
from turbo_dllm_amd import options

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,kept,reduction,postpone,device_count", [
    (1, 1, "mean", True, False),
    (63, 63, "sum", True, False),            # all rows, no map of rows
    (300, 0, "mean", True, False),           # no row with a loss
    (300, 1, "mean", True, False),
    (1030, 257, "none", True, False),        # one row past a tile
    (1030, 700, "mean", False, False),       # float32 accumulator
    (4097, 513, "sum", True, True),          # more rows to clear than one workgroup takes
    (700, 0, "mean", True, True),
    (1500, 900, "mean", False, True),        # blocks of rows, the last ones empty
])
def test_joined_launches(gpu_device, n, kept, reduction, postpone, device_count):
    print("[case]", n, kept, reduction, postpone, device_count, flush=True)
    h, v = 128, 1024
    gen = torch.Generator().manual_seed(n)
    hidden = torch.randn(n, h, generator=gen).bfloat16().to(gpu_device)
    weight = (torch.randn(v, h, generator=gen) * 0.1).bfloat16().to(gpu_device)
    labels = torch.randint(0, v, (n,), generator=gen)
    labels[torch.randperm(n, generator=gen)[kept:]] = -100
    labels = labels.to(gpu_device)
    mode = "device" if device_count else "sync"
    rows, targets, _, row_idx, count, m = native.compact_loss_rows(hidden, labels, None, -100, mode)
    rows, targets = rows[:m], targets[:m]
    count = count if device_count else None
    go = (torch.rand(n if reduction == "none" else 1, generator=gen) + 0.5).to(gpu_device)
    common = dict(ignore_index=-100, exclude_index=7, logit_softcap=0.0, compute_weight_grad=True,
                  postpone_weight_grad=postpone, row_idx=row_idx, n_out=n, row_count=count)
    with options.panel_budget(0 if postpone else 512 * v * 2):
        panel = options.get_panel_bytes()
        losses, _, valid, dh32, dw32 = native.forward_with_gradients(rows, weight, targets, **common)
        dh, dw = native.apply_grad_output(
            dh32, None if postpone else dw32, go, valid, reduction=reduction,
            dtype=torch.bfloat16, row_idx=row_idx, n_out=n, vocab=v, row_count=count)
        if postpone:
            dw = native.grad_weight_from_panel(
                rows, dw32, go, valid, reduction=reduction, vocab=v, panel_bytes=panel,
                row_count=count, row_idx=row_idx, n_out=n)
        loss, valid2, dh32, dw32, row_of = native.forward_with_gradients_reduced(
            rows, weight, targets, reduction=reduction, **common)
        for _ in range(2):   # a second backward on the same workspace
            dh2, dw2 = native.finish_gradients(
                dh32, dw32, go, valid2, reduction=reduction, n_out=n, vocab=v, row_of=row_of,
                row_count=count, rows=rows if postpone else None, panel_bytes=panel)
            assert torch.equal(dh, dh2) and torch.equal(dw, dw2)
    assert float(valid) == float(valid2) == float((labels != -100).sum())
    if reduction == "none":
        assert torch.equal(loss, losses)
    else:
        want = losses.double().sum() / (valid.double() if reduction == "mean" else 1.0)
        want = want.reshape(())
        if reduction == "mean" and kept == 0:
            assert bool(loss.isnan()) and bool(want.isnan())
        else:
            assert abs(float(loss) - float(want)) <= n * 2.0 ** -24 * abs(float(want))


@pytest.mark.parametrize("n,kept", [(1, 0), (1, 1), (37, 20), (256, 1), (256, 255), (256, 256)])
@pytest.mark.parametrize("reduction,trainable", [("mean", True), ("none", True), ("none", False)])
def test_rows_of_one_tile_are_not_compacted(gpu_device, n, kept, reduction, trainable):
    """Against the same call on the compacted rows; whatever ignored rows and their upstream
    gradients hold stays out of the results.  (Both calls make the same products; sums over the
    rows meet zeros in between: bit for bit.)"""
    from turbo_dllm_amd.tiled_linear_cross_entropy import tiled_linear_cross_entropy
    print("[case]", n, kept, reduction, trainable, flush=True)
    h, v = 192, 1600
    gen = torch.Generator().manual_seed(n + kept)
    hidden = torch.randn(n, h, generator=gen).bfloat16()
    weight = (torch.randn(v, h, generator=gen) * 0.1).bfloat16().to(gpu_device)
    labels = torch.randint(0, v, (n,), generator=gen)
    gone = torch.randperm(n, generator=gen)[kept:]
    labels[gone] = -100
    hidden[gone] = float("nan")
    up = torch.rand(n, generator=gen) + 0.5
    up[gone] = float("inf")
    keep = (labels != -100).nonzero().flatten()

    def step(x, y, go, mode):
        x = x.to(gpu_device).requires_grad_()
        w = weight.clone().requires_grad_(trainable)
        with torch.no_grad():
            alone = tiled_linear_cross_entropy(x, w, y.to(gpu_device), reduction="none")
        loss = tiled_linear_cross_entropy(x, w, y.to(gpu_device), reduction=reduction,
                                          compaction=mode)
        loss.backward(go.to(gpu_device) if reduction == "none" else torch.ones_like(loss))
        return alone, loss.detach(), x.grad, w.grad

    alone, loss, dx, dw = step(hidden, labels, up, "sync")
    rows = keep.to(gpu_device)
    assert not alone.isnan().any() and bool((alone[gone.to(gpu_device)] == 0).all())
    assert bool((dx[gone.to(gpu_device)] == 0).all())
    if kept == 0:
        assert bool(loss.isnan().all()) == (reduction == "mean") and bool((dx == 0).all())
        assert not trainable or bool((dw == 0).all())
        return
    _, want, want_dx, want_dw = step(hidden[keep], labels[keep], up[keep], "none")
    assert torch.equal(loss[rows] if reduction == "none" else loss, want) or (
        reduction == "mean" and abs(float(loss - want)) <= n * 2.0 ** -24 * float(want))
    assert torch.equal(dx[rows], want_dx)
    # grad_weight's sum over rows is taken 32 at a time, in other places of the groups
    if trainable:
        assert float((dw.double() - want_dw.double()).norm()) <= 4e-3 * float(want_dw.double().norm())


@pytest.mark.parametrize("b,t,kept,dtype", [
    (1, 5, 5, torch.bfloat16), (3, 300, 1, torch.bfloat16), (4, 257, 300, torch.bfloat16),
    (7, 65, 64, torch.float32),
])
def test_gathered_sample_rows(gpu_device, b, t, kept, dtype):
    """Rows, targets and per-row factors of a batch in one launch: bit for bit what the
    separate operations make, and padded to 64 rows with zeros and ignored labels."""
    gen = torch.Generator().manual_seed(b * t)
    hidden = torch.randn(b * t, 96, generator=gen).to(dtype).to(gpu_device)
    labels = torch.randint(0, 1000, (b, t), generator=gen).to(gpu_device)
    weights = torch.rand(b, t, generator=gen).to(gpu_device)
    counts = torch.rand(b, generator=gen).to(gpu_device) * 9
    mask = torch.zeros(b * t, dtype=torch.bool)
    mask[torch.randperm(b * t, generator=gen)[:kept]] = True
    mask = mask.to(gpu_device)
    row_idx, count = native.compact_mask_device(mask)
    rows, targets, factors = native.gather_sample_rows(hidden, labels, weights, counts, t, row_idx,
                                                       count, kept)
    at = mask.nonzero().flatten()
    want = weights.flatten()[at] / ((counts[at // t] + 1.0e-5) * b)
    assert torch.equal(rows[:kept], hidden[at]) and torch.equal(targets[:kept], labels.flatten()[at])
    assert torch.equal(factors[:kept], want)
    assert len(rows) == -(-kept // 64) * 64
    assert bool((rows[kept:] == 0).all()) and bool((targets[kept:] == -100).all())
