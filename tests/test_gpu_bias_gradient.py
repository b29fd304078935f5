"""The bias in the logit-gradient panel of the direct engine and its gradient's row sums.

Its gradient is a float32 sum of float32 logit gradients, rounded once to the input type:
2^-8 of an entry at most in bf16, 2^-11 in f16.  Before that a logit is off by sqrt(H) * 2^-24
of its largest partial sum as a random walk (about 20 here: 4e-5 at H = 1024), and an entry by
as much relative to itself."""

import pytest
import torch

from turbo_dllm_amd.tiled_linear_cross_entropy import tiled_linear_cross_entropy


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("m,h,v,cap,exclude,compaction", [
    (1, 64, 256, 0.0, False, "sync"),
    (257, 128, 257, 0.0, True, "sync"),       # one row and one word past a tile
    (300, 1024, 5000, 20.0, True, "sync"),
    (640, 328, 8200, 0.0, False, "device"),   # hidden size with a column tail
])
def test_gradient_of_the_bias(gpu_device, m, h, v, cap, exclude, compaction, dtype):
    print("[case]", m, h, v, cap, exclude, compaction, dtype, flush=True)
    gen = torch.Generator().manual_seed(m + v)
    weight = (torch.randn(v, h, generator=gen) * 0.05).to(dtype).to(gpu_device)
    hidden = torch.randn(m, h, generator=gen).to(dtype).to(gpu_device).requires_grad_()
    bias = (torch.randn(v, generator=gen) * 0.5).to(dtype).to(gpu_device).requires_grad_()
    labels = torch.randint(0, v - 1, (m,), generator=gen).to(gpu_device)
    if compaction == "device":
        labels[::3] = -100
    tiled_linear_cross_entropy(hidden, weight, labels, bias=bias, reduction="sum", dtype=dtype,
                               logit_softcap=cap, compaction=compaction,
                               exclude_index=v - 1 if exclude else None).backward()
    b64 = bias.detach().double().requires_grad_()
    z = hidden.detach().double() @ weight.double().t() + b64
    if cap:
        z = cap * torch.tanh(z / cap)
    if exclude:
        z = z.index_fill(1, torch.tensor([v - 1], device=z.device), float("-inf"))
    torch.nn.functional.cross_entropy(z, labels, reduction="sum").backward()
    bar = (2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -11) + 4e-5
    assert float((bias.grad.double() - b64.grad).norm() / b64.grad.norm()) <= bar
