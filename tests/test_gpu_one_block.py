"""Reduced losses whose rows take one block although their panel is larger than the default
(``reduced_loss_panel_bytes``): the gradient of the head waits for the backward instead of being
summed in float32 over two blocks."""

import pytest
import torch

from turbo_dllm_amd import _lib, options
from turbo_dllm_amd import chunked_linear_ce_native as native
from turbo_dllm_amd.loss import masked_token_loss
from turbo_dllm_amd.tiled_linear_cross_entropy import tiled_linear_cross_entropy

DEFAULT = 5 << 29


def test_where_one_block_is_taken():
    """Panels above the default, up to the default and one 16-bit gradient of the head."""
    size = _lib.library().tlce_reduced_loss_panel_bytes
    tile = 256 * 262144 * 2
    fits = DEFAULT // tile                                      # 20 token tiles
    for h, extra in ((64, 0), (320, 1), (3840, 15)):
        assert DEFAULT + 2 * 262144 * h >= (fits + extra) * tile
        assert size(256 * fits, h, 262144, _lib.DTYPE_BF16) == 0
        for tiles in range(fits + 1, fits + 18):
            want = tiles * tile if tiles <= fits + extra else 0
            assert size(256 * tiles, h, 262144, _lib.DTYPE_BF16) == want
            assert size(256 * tiles - 255, h, 262144, _lib.DTYPE_BF16) == want
            if want:
                plan = _lib.query_fused_plan(256 * tiles, h, 262144, _lib.DTYPE_BF16, want)
                assert plan["n_blocks"] == 1 and plan["block_rows"] == 256 * tiles
    assert size(6000, 4096, 262144, _lib.DTYPE_F16) == 0        # not formed in the forward
    assert size(6000, 4096, 262143, _lib.DTYPE_BF16) == 0
    assert size(0, 4096, 262144, _lib.DTYPE_BF16) == 0
    with options.panel_budget(1 << 30):                         # a budget that was asked for
        assert native.reduced_loss_panel_bytes(6000, 4096, 262144, torch.bfloat16) == 1 << 30


@pytest.mark.gpu
@pytest.mark.parametrize("loss_kind", ["ce", "masked"])
def test_one_block_beyond_the_default(gpu_device, loss_kind):
    m, h, v = 5300, 320, 262144                                 # 21 token tiles
    print("[case]", loss_kind, m, h, v, flush=True)
    gen = torch.Generator(device=gpu_device).manual_seed(5)
    hidden = torch.randn(m, h, generator=gen, device=gpu_device).bfloat16()
    weight = (torch.randn(v, h, generator=gen, device=gpu_device) * 0.05).bfloat16()
    labels = torch.randint(0, v, (m,), generator=gen, device=gpu_device)
    weights = torch.rand(m, generator=gen, device=gpu_device)
    head = torch.nn.Linear(h, v, bias=False, device="meta")

    def step():
        x = hidden.clone().requires_grad_()
        w = torch.nn.Parameter(weight.clone())
        with _lib.kernel_profile() as prof:
            if loss_kind == "ce":
                loss = tiled_linear_cross_entropy(x, w, labels, dtype=torch.bfloat16)
            else:
                head.weight = w
                loss = masked_token_loss(x, labels, weights, head, valid_token_count=float(m))
        loss.backward()
        return prof.launches, [loss.detach(), x.grad, w.grad]

    launches, one = step()
    assert launches["exp_logits_panel"] == 2 and launches["grad_weight_gemm"] == 0
    with options.panel_budget(DEFAULT):
        launches, two = step()
    assert launches["exp_logits_panel"] == 4 and launches["grad_weight_gemm"] == 2
    # The same entries and grad_hidden.  grad_weight is rounded on either side where its hidden
    # rows take their factor (with the upstream gradient or without) and at the end: four
    # independent roundings of 1.66e-3, 3.32e-3, and 8 % for the spread of one sample.
    for a, b, bound in zip(one, two, (1e-6, 1e-4, 3.6e-3)):
        error = float((a.double() - b.double()).norm() / b.double().norm())
        print("[case] differs by", error, flush=True)
        assert error <= bound
