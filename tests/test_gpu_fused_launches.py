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
