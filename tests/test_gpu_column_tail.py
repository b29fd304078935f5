"""16-bit heads whose hidden size is a multiple of 8 but not of 64 on the direct engine: the
last K tile of the logits contraction comes from zero-padded copies of the last columns.

Losses are float32 sums of exact products (1e-5); gradients round the logit gradients and the
result to the input type, 2-norm sqrt(2) * 2^-7 / sqrt(12) * sqrt(3 / (8 ln 2)) = 2.35e-3 in
bf16 (an eighth of it in f16, whose smallest logit gradients are subnormal here: held to the
bf16 bar), and 10 % for the spread of one sample."""

import pytest
import torch

from turbo_dllm_amd import _lib
from turbo_dllm_amd.streaming_soft_embedding import streaming_soft_embedding
from turbo_dllm_amd.tiled_linear_cross_entropy import tiled_linear_cross_entropy

BAR = 1.1 * 2.35e-3


def operands(dev, m, h, v, dtype, seed):
    gen = torch.Generator().manual_seed(seed)
    weight = (torch.randn(v, h, generator=gen) * 0.05).to(dtype)
    labels = torch.randint(0, v - 1, (m,), generator=gen)
    hidden = torch.randn(m, h, generator=gen) + weight[labels].float() * (6.0 / (0.05 ** 2 * h))
    return hidden.to(dtype).to(dev), weight.to(dev), labels.to(dev)


def off(got, want):
    return float((got.double() - want).norm() / want.norm())


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("m,h,v,kw", [
    (300, 264, 7001, {}),                                    # one piece in the last tile
    (65, 312, 33000, dict(logit_softcap=20.0)),              # all but one of its eight
    (257, 328, 8200, dict(exclude_index=8199, bias=True)),
    (520, 1000, 4096, dict(compaction="device")),
])
def test_against_float64(gpu_device, m, h, v, kw, dtype):
    print("[case]", m, h, v, kw, dtype, flush=True)
    kw = dict(kw)
    assert _lib.query_plan(m, h, v, _lib.DTYPE_BF16, True)["engine"] == "mfma_direct"
    hidden, weight, labels = operands(gpu_device, m, h, v, dtype, m + h)
    bias = None
    if kw.pop("bias", False):
        bias = (torch.randn(v, generator=torch.Generator().manual_seed(1)) * 0.1).to(dtype).to(gpu_device)
    if "compaction" in kw:
        labels[::3] = -100
    excluded = kw.get("exclude_index")
    x, w = hidden.clone().requires_grad_(), weight.clone().requires_grad_()
    if excluded is not None:
        # an excluded word may hold anything: it must reach no neighbour's tile
        with torch.no_grad():
            w[excluded] = float("nan")
    b = None if bias is None else bias.clone().requires_grad_()
    loss = tiled_linear_cross_entropy(x, w, labels, bias=b, reduction="sum", dtype=dtype, **kw)
    loss.backward()
    x64, w64 = hidden.double().requires_grad_(), weight.double().requires_grad_()
    z = x64 @ w64.t()
    if bias is not None:
        z = z + bias.double()
    if "logit_softcap" in kw:
        z = kw["logit_softcap"] * torch.tanh(z / kw["logit_softcap"])
    if excluded is not None:
        z = z.index_fill(1, torch.tensor([excluded], device=z.device), float("-inf"))
    want = torch.nn.functional.cross_entropy(z, labels, reduction="sum")
    want.backward()
    assert abs(float(loss.detach()) - float(want)) <= 1e-5 * float(want)
    keep = torch.arange(v, device=gpu_device) != (-1 if excluded is None else excluded)
    if excluded is None:   # (0 times the excluded word's NaN is what its rows' gradient gets)
        assert off(x.grad, x64.grad) <= BAR
    assert off(w.grad[keep], w64.grad[keep]) <= BAR


@pytest.mark.gpu
def test_soft_embedding(gpu_device):
    hidden, weight, _ = operands(gpu_device, 300, 264, 9000, torch.bfloat16, 2)
    got = streaming_soft_embedding(hidden, weight, row_chunk_size=64, vocab_chunk_size=1024)
    want = (hidden.double() @ weight.double().t()).softmax(1) @ weight.double()
    assert off(got, want) <= BAR


def test_small_calls_keep_the_staged_engine():
    plan = lambda m, h, v: _lib.query_plan(m, h, v, _lib.DTYPE_BF16, True)["engine"]
    assert plan(300, 264, 7001) == "mfma_direct" and plan(300, 64, 7001) == "mfma_direct"
    assert plan(300, 264, 1000) == plan(64, 264, 70000) == plan(300, 248, 70000) == "mfma"
    lib = _lib.library()
    size = lib.tlce_forward_workspace_bytes(300, 264, 7001, _lib.DTYPE_BF16)
    assert size >= (7001 * 64 + 300 * 320) * 2          # the copies
