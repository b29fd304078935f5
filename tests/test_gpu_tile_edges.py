"""The tile engines and their launch shapes at the sizes where they can go wrong: one,
two and three K steps (the main loop peels its first and its last two), rows and
vocabularies around tile edges, and tile counts that do not divide into groups of four.
Loss within 1e-3 relative and gradients within 2e-2 relative max-norm of the float32
oracle for 16-bit inputs, the operator's bars."""

import pytest
import torch

import linear_ce_oracle as oracle
from turbo_dllm_amd import options
from turbo_dllm_amd.tiled_linear_cross_entropy import tiled_linear_cross_entropy

pytestmark = pytest.mark.gpu


def check(dev, m, h, v, dtype, mode, seed=5, **kw):
    print("[case]", m, h, v, dtype, mode, kw, flush=True)
    gen = torch.Generator().manual_seed(seed)
    hidden = torch.randn(m, h, generator=gen).to(dtype)
    weight = (torch.randn(v, h, generator=gen) * 0.05).to(dtype)
    labels = torch.randint(0, v, (m,), generator=gen)
    x = hidden.to(dev).requires_grad_(True)
    w = weight.to(dev).requires_grad_(True)
    with options.gradient_mode(mode):
        loss = tiled_linear_cross_entropy(x, w, labels.to(dev), dtype=dtype, **kw)
        loss.backward()
    torch.cuda.synchronize()
    ref = oracle.dense_linear_ce(hidden, weight, labels, dtype=torch.float32, **kw)
    dh, dw, _ = oracle.dense_linear_ce_grads(hidden, weight, labels, dtype=torch.float32, **kw)
    rtol, gtol = (2e-5, 3e-5) if dtype == torch.float32 else (1e-3, 2e-2)
    err_h = oracle.relative_max_error(x.grad, dh)
    err_w = oracle.relative_max_error(w.grad, dw)
    print("[case] errors", float(loss.detach()), float(ref), err_h, err_w, flush=True)
    assert abs(float(loss.detach()) - float(ref)) <= rtol * abs(float(ref))
    assert err_h <= gtol and err_w <= gtol


@pytest.mark.parametrize("mode", options.GRADIENT_MODES)
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("m,h,v", [
    (1, 64, 64),            # one K step, one row
    (64, 128, 320),         # two K steps, one 64-row K slab for grad_weight
    (129, 192, 256),        # three K steps; two and a remainder of token rows
    (255, 256, 257 + 63),   # a row short of a tile, one vocabulary row past one
    (257, 320, 512),        # a row past a tile
    (1153, 64, 1088),       # five token tiles (groups of 3 and 2), five vocabulary tiles
    (2100, 1152, 448),      # nine token tiles and five hidden tiles
])
def test_direct_engine_edges(gpu_device, m, h, v, dtype, mode):
    check(gpu_device, m, h, v, dtype, mode)


@pytest.mark.parametrize("mode", options.GRADIENT_MODES)
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("m,h,v,kw", [
    (1, 64, 2, {}),                                 # the tail is the whole K range
    (65, 64, 63, {}),                               # and holds all but one of its rows
    (130, 128, 65, dict(exclude_index=64)),         # one slab and a tail of one row
    (257, 192, 191, {}),                            # two slabs and a tail
    (300, 256, 4099, dict(logit_softcap=20.0)),     # the tail in the last of the K splits
    (1030, 320, 32003, {}),                         # two panels of the recomputing backward
])
def test_direct_engine_ragged_vocabularies(gpu_device, m, h, v, kw, dtype, mode):
    """Vocabularies (K of the grad_hidden contraction) and row counts (K of grad_weight)
    that end inside a 64-row K slab, in the recomputing backward, which such heads take in
    either mode."""
    with options.panel_budget((32 << 20) if v > 30000 and mode == "recompute" else 0):
        check(gpu_device, m, h, v, dtype, mode, **kw)


@pytest.mark.parametrize("m,h,v,kw", [
    (1, 4, 64, {}),                                 # one piece of one K stage
    (3, 4, 63, {}),                                 # the last vocabulary of the generic engine
    (31, 36, 127, dict(logit_softcap=30.0)),        # a K stage and a remainder
    (128, 32, 128, {}),                             # whole tiles, one K stage
    (129, 100, 257, dict(exclude_index=7)),         # a row and a vocabulary row past tiles
    (260, 260, 3001, {}),                           # K splits of grad_hidden, odd vocabulary
    (700, 64, 4099, dict(logit_softcap=20.0)),
])
def test_float32_engine_edges(gpu_device, m, h, v, kw):
    check(gpu_device, m, h, v, torch.float32, "recompute", **kw)


def test_float32_engine_with_bias_matches_the_oracle(gpu_device):
    gen = torch.Generator().manual_seed(3)
    m, h, v = 130, 68, 300
    hidden = torch.randn(m, h, generator=gen)
    weight = torch.randn(v, h, generator=gen) * 0.05
    bias = torch.randn(v, generator=gen) * 0.1
    labels = torch.randint(0, v, (m,), generator=gen)
    leaves = [t.to(gpu_device).requires_grad_(True) for t in (hidden, weight, bias)]
    loss = tiled_linear_cross_entropy(leaves[0], leaves[1], labels.to(gpu_device),
                                      bias=leaves[2], dtype=torch.float32)
    loss.backward()
    ref = [t.clone().requires_grad_(True) for t in (hidden, weight, bias)]
    expected = torch.nn.functional.cross_entropy(ref[0] @ ref[1].t() + ref[2], labels)
    expected.backward()
    assert abs(float(loss.detach()) - float(expected.detach())) <= 2e-5 * float(expected.detach())
    for got, want in zip(leaves, ref):
        assert oracle.relative_max_error(got.grad, want.grad) <= 3e-5
