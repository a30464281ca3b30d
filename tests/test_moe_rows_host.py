"""Host side of the MoE down stage by way of rows: when scratch is asked for, how much, and what happens when there is none (no GPU)."""

import types

import pytest
import torch

from flydsl_amd import _lib

BF16, FP16, F32 = 0, 1, 2


def _bytes(tokens, topk, sorted_size, model, out=BF16, mx=0):
    """mx: 0 one scale per row, 1 the MX pair, 2 int4 weights."""
    return _lib.lib().psg_moe_rows_workspace_bytes(tokens, topk, sorted_size, model, out, mx)


def _layout(tokens, topk, sorted_size, model):
    up = lambda v: (v + 15) // 16 * 16
    return up(sorted_size * model * 2) + up((tokens + 1) * 4) + up(tokens * topk * 4) + sorted_size * 4


@pytest.mark.parametrize("mx", [0, 1])
@pytest.mark.parametrize("tokens,topk,model", [(4096, 8, 4096), (1023, 6, 2304), (513, 5, 7168)])
def test_scratch_holds_the_rows_and_the_lists(tokens, topk, model, mx):
    size = tokens * topk + 32 * 128 - topk
    assert _bytes(tokens, topk, size, model, mx=mx) == _bytes(tokens, topk, size, model, FP16, mx) == _layout(tokens, topk, size, model)


def test_scratch_starts_and_ends_where_the_rule_says():
    mb = 1 << 20
    for mx, least, most in ((1, 12 * mb, 4 << 30), (0, 24 * mb, 1 << 30), (2, 24 * mb, 256 * mb)):
        # topk * model * 2 = 64 KiB of additions a token
        least_tokens = least >> 16
        assert _bytes(least_tokens, 8, least_tokens * 8, 4096, mx=mx) > 0
        assert _bytes(least_tokens - 1, 8, least_tokens * 8, 4096, mx=mx) == 0
        # the bound counts the whole buffer: rows of padding too
        size = next(s for s in range(most // 8192, 0, -1) if _layout(4096, 8, s, 4096) <= most)
        assert _bytes(4096, 8, size, 4096, mx=mx) == _layout(4096, 8, size, 4096) <= most
        assert _bytes(4096, 8, size + 1, 4096, mx=mx) == 0
    assert _bytes(32768, 8, 32768 * 8 + 32 * 128, 7168) == 0
    assert _bytes(65536, 3, 65536 * 3, 1024) == 0 < _bytes(65536, 3, 65536 * 3, 1024, mx=1)  # few slots: adding directly
    assert _bytes(4096, 8, 40000, 4096, F32) == 0


@pytest.fixture
def gpu(monkeypatch):
    """call_scratch's surroundings: current stream 7, nothing captured, an allocator with `room` bytes."""
    g = types.SimpleNamespace(room=1 << 20, stream=7, capturing=False, asked=[])

    def empty(n, **kw):
        g.asked.append(n)
        if n > g.room:
            raise torch.cuda.OutOfMemoryError("no room")
        return ("buffer", n)

    monkeypatch.setattr(torch.cuda, "current_stream", lambda d=None: types.SimpleNamespace(cuda_stream=g.stream))
    monkeypatch.setattr(torch, "empty", empty)
    monkeypatch.setattr(_lib, "_torch_capturing", lambda: g.capturing)
    monkeypatch.setattr(_lib, "_refused", {})
    return g


def test_call_scratch_allocates_on_the_current_stream_only(gpu):
    assert _lib.call_scratch("cuda:0", 100, 7) == ("buffer", 100)
    assert _lib.call_scratch("cuda:0", 100, 8) is None  # another stream: its work is not ordered with this memory's next owner
    assert _lib.call_scratch("cuda:0", 0, 7) is None
    gpu.capturing = True
    assert _lib.call_scratch("cuda:0", 100, 7) is None
    assert gpu.asked == [100]


def test_call_scratch_remembers_a_refusal(gpu):
    assert _lib.call_scratch("cuda:0", 2 << 20, 7) is None
    for _ in range(_lib._REFUSED_CALLS):
        assert _lib.call_scratch("cuda:0", 2 << 20, 7) is None
    assert gpu.asked == [2 << 20]  # one failing allocation in all these calls
    assert _lib.call_scratch("cuda:0", 1 << 20, 7) == ("buffer", 1 << 20)  # less is still asked for
    assert _lib.call_scratch("cuda:1", 2 << 20, 7) is None and gpu.asked[-1] == 2 << 20  # another device is another matter
    gpu.room = 4 << 20
    assert _lib.call_scratch("cuda:0", 2 << 20, 7) == ("buffer", 2 << 20)  # and in the end the allocator is asked again
    assert _lib.call_scratch("cuda:0", 3 << 20, 7) == ("buffer", 3 << 20)
