"""Last token tiles of at most 64 and at most 128 rows, which run narrower than 256 (engine
``NarrowEngine``): one to four K steps, rows around both widths, alone and after a whole tile, a
vocabulary that ends inside a tile and inside a K slab.  Per-token losses are those of the same rows
in a tile of 256, bit for bit (the sums run in the same order), where the forward has narrow tiles:
exponentiated logits, of bf16 over whole K slabs.  Others run narrow in grad_hidden only.  Gradients
within the operator's 2e-2 relative max-norm of the float32 oracle."""

import pytest
import torch

import linear_ce_oracle as oracle
from turbo_dllm_amd import _lib
from turbo_dllm_amd import chunked_linear_ce_native as native
from turbo_dllm_amd.tiled_linear_cross_entropy import tiled_linear_cross_entropy

pytestmark = pytest.mark.gpu


def step(hidden, weight, labels, reduction, trainable, **keywords):
    x = hidden.clone().requires_grad_()
    w = weight.clone().requires_grad_(trainable)
    loss = tiled_linear_cross_entropy(x, w, labels, reduction=reduction, dtype=x.dtype, **keywords)
    loss.sum().backward()
    return loss.detach(), x.grad, w.grad


@pytest.mark.parametrize("rows", [1, 16, 63, 64, 65, 127, 128, 129])
@pytest.mark.parametrize("before", [0, 256])
@pytest.mark.parametrize("h,v,keywords", [
    (64, 320, {}),
    (128, 448, dict(logit_softcap=20.0)),
    (192, 1088, dict(exclude_index=300)),
    (256, 4096, {}),
    (320, 515, {}),
])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_last_tiles(gpu_device, rows, before, h, v, keywords, dtype):
    m, wide = before + rows, before + 200
    print("[case]", m, h, v, keywords, dtype, flush=True)
    gen = torch.Generator().manual_seed(m + h + v)
    hidden = torch.randn(wide, h, generator=gen).to(dtype)
    weight = (torch.randn(v, h, generator=gen) * 0.05).to(dtype)
    labels = torch.randint(0, 300, (wide,), generator=gen)
    on_gpu = [t.to(gpu_device) for t in (hidden, weight, labels)]
    if native.fused_gradients_supported(on_gpu[0], on_gpu[1], None, False):
        with _lib.kernel_profile() as prof:
            losses, _, _ = step(on_gpu[0][:m], on_gpu[1], on_gpu[2][:m], "none", False, **keywords)
        assert prof.launches["exp_logits_panel"] > 0
        in_wide, _, _ = step(*on_gpu, "none", False, **keywords)
        assert torch.equal(losses, in_wide[:m])
    else:
        assert dtype == torch.float16 or v % 64 != 0
    _, grad_hidden, grad_weight = step(on_gpu[0][:m], on_gpu[1], on_gpu[2][:m], "mean", True,
                                       **keywords)
    want_hidden, want_weight, _ = oracle.dense_linear_ce_grads(
        hidden[:m], weight, labels[:m], dtype=torch.float32, **keywords)
    assert oracle.relative_max_error(grad_hidden, want_hidden) <= 2e-2
    assert oracle.relative_max_error(grad_weight, want_weight) <= 2e-2


@pytest.mark.parametrize("m", [8300, 8448, 8704])
def test_grad_hidden_in_chunks_of_one_round(gpu_device, monkeypatch, m):
    """15 x 33 and 15 x 34 tiles of grad_hidden, unsplit, of rows whose number the host knows: two
    chunks of 17 token tiles, the last one ragged.  Within the operator's 2e-2 relative max-norm of
    float32."""
    h, v = 3840, 512
    inner = native.forward_with_gradients_reduced

    def counted(*args, row_count=None, **others):
        assert row_count is None
        calls.append(_lib.query_fused_plan(m, h, v, _lib.DTYPE_BF16, 0))
        return inner(*args, **others)

    calls = []
    monkeypatch.setattr(native, "forward_with_gradients_reduced", counted)
    gen = torch.Generator(device=gpu_device).manual_seed(m)
    hidden = torch.randn(m, h, generator=gen, device=gpu_device).bfloat16()
    weight = (torch.randn(v, h, generator=gen, device=gpu_device) * 0.02).bfloat16()
    labels = torch.randint(0, v, (m,), generator=gen, device=gpu_device)
    _, grad_hidden, _ = step(hidden, weight, labels, "sum", True, compaction="none")
    assert [(plan["n_blocks"], plan["grad_hidden_k_splits"]) for plan in calls] == [(1, 1)]
    p = torch.softmax(hidden.float() @ weight.float().t(), 1)
    p[torch.arange(m, device=gpu_device), labels] -= 1.0
    want = p @ weight.float()
    assert oracle.relative_max_error(grad_hidden, want) <= 2e-2
    assert (grad_hidden.float() - want).norm(dim=1).div(want.norm(dim=1)).max() <= 2e-2
