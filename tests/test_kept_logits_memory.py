"""How much memory ``kept_logits_buffer`` takes of what is left: an eighth, a twenty-fourth of the
device, and nothing that the backward's own workspace and gradients need.  The library's size
queries run on the host; what the allocator would answer is given."""

import pytest
import torch
import torch.utils.checkpoint

from turbo_dllm_amd import _lib
from turbo_dllm_amd import chunked_linear_ce_native as native

M, H, V = 512, 1024, 5000                       # 2 x 20 tiles
COLUMN = 2 * 256 * 256 * 4                      # of token tiles, per vocabulary tile
MIB, GIB = 1 << 20, 1 << 30


def backward_needs(n_out):
    return (_lib.library().tlce_backward_workspace_bytes(M, H, V, _lib.DTYPE_BF16, 1, 0, 0)
            + (n_out + V) * H * 2)


def buffer(monkeypatch, left, total=288 * GIB, n_out=M, cached=0, unasked=0):
    monkeypatch.setattr(native, "_KEEP_UNASKED_BYTES", unasked)
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: False)
    monkeypatch.setattr(torch.cuda, "mem_get_info", lambda device: (left - cached, total))
    monkeypatch.setattr(native, "_memory_cached", lambda device: cached)
    rows = torch.empty(M, H, dtype=torch.bfloat16)
    kept = native.kept_logits_buffer(M, rows, V, None, n_out)
    return 0 if kept is None else kept.numel()


def test_what_is_taken_of_the_memory_left(monkeypatch):
    need = backward_needs(M)
    assert buffer(monkeypatch, 8 * GIB) == 20 * COLUMN                  # all logits
    assert buffer(monkeypatch, 8 * 7 * COLUMN + need) >= 7 * COLUMN     # an eighth
    for left in (need + 3 * COLUMN, 8 * 11 * COLUMN, 8 * 19 * COLUMN + 5):
        want = min(left // 8, left - need, 20 * COLUMN) // COLUMN * COLUMN
        assert buffer(monkeypatch, left) == max(want, 0)
        assert buffer(monkeypatch, left, cached=left - MIB) == max(want, 0)
    assert buffer(monkeypatch, 8 * GIB, total=24 * 5 * COLUMN) == 5 * COLUMN
    for left in (0, MIB, need, need + COLUMN - 1):                      # the backward alone
        assert buffer(monkeypatch, left) == 0
    assert buffer(monkeypatch, 0, unasked=20 * COLUMN) == 20 * COLUMN   # small: not asked
    assert buffer(monkeypatch, 0, unasked=20 * COLUMN - 1) == 0
    # un-compacted gradients count as they are: 100 000 rows, 205 MB
    assert buffer(monkeypatch, backward_needs(100_000), n_out=100_000) == 0


def test_a_backward_without_memory_gives_the_logits_back():
    kept = torch.empty(4096, dtype=torch.uint8)
    tried = []

    def call(buffer):
        tried.append(buffer)
        if buffer is not None:
            raise torch.OutOfMemoryError("no room beside the logits")
        return "recomputed"

    assert native.from_kept_logits(kept, call) == "recomputed"
    assert tried == [kept, None] and kept.untyped_storage().size() == 0
    assert native.from_kept_logits(kept, call) == "recomputed"          # a retained graph
    assert tried[2:] == [None]
    with pytest.raises(ValueError):                                     # other errors pass
        native.from_kept_logits(torch.empty(8), lambda buffer: (_ for _ in ()).throw(ValueError))


def test_what_each_allocator_holds(monkeypatch):
    def stats(device):
        if backend == "pluggable":
            raise RuntimeError("CUDAPluggableAllocator does not yet support getDeviceStats.")
        current = {"reserved_bytes": 100, "active_bytes": 60, "inactive_split_bytes": 30}
        return {name: {"all": {"current": n}} for name, n in current.items()} if used else {}

    monkeypatch.setattr(torch.cuda, "memory_stats_as_nested_dict", stats)
    monkeypatch.setattr(torch.cuda, "get_allocator_backend", lambda: backend)
    for backend, used, want in (("native", True, 10), ("native", False, 0), ("pluggable", True, 0)):
        assert native._memory_cached(torch.device("cuda:0")) == want


def test_nothing_is_kept_where_saved_tensors_are_packed(monkeypatch):
    assert buffer(monkeypatch, 8 * GIB) > 0
    with torch.autograd.graph.save_on_cpu():
        assert buffer(monkeypatch, 8 * GIB) == 0
    seen = []

    def layer(x):
        seen.append(buffer(monkeypatch, 8 * GIB))
        return x.sin()

    x = torch.ones(3, requires_grad=True)
    torch.utils.checkpoint.checkpoint(layer, x, use_reentrant=False).sum().backward()
    assert seen == [0, 0] and buffer(monkeypatch, 8 * GIB) > 0
    monkeypatch.delattr(torch._C._autograd, "_top_saved_tensors_default_hooks")
    assert buffer(monkeypatch, 8 * GIB) == 0
