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
