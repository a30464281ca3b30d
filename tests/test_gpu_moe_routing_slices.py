"""Gating and sorting of more than 4096 pairs with a workspace: the gating inside the first launch (slices of one, two and four wavefronts' tokens, of two
passes), in a launch of its own where a slice would be a longer chain, and the offsets worked out in the last launch or, beyond 1024 experts, in one of
their own.  All of it must equal the gating kernel followed by the sorter in its single launch."""

import pytest
import torch

pytestmark = pytest.mark.gpu


def _outputs(tokens, topk, experts, block):
    from flydsl_amd.kernels.moe.moe_sorting import sorted_sizes

    rows = sorted_sizes(tokens, topk, experts, block)[0] + 5
    return [torch.full((n,), 77, dtype=dt, device="cuda") for n, dt in ((rows, torch.int32), (rows, torch.float32), ((rows + block - 1) // block, torch.int32), (2, torch.int32))]


@pytest.mark.parametrize("masked", [False, True])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("tokens,experts,topk,block", [
    (513, 32, 8, 128), (4096, 32, 8, 128), (8193, 17, 1, 64),     # one wavefront's tokens a slice; a token more than whole slices; one slot
    (4100, 33, 6, 32), (3001, 64, 6, 128), (2049, 32, 4, 16),     # two and four wavefronts
    (6000, 32, 1, 64), (4098, 256, 4, 32), (3000, 128, 2, 64),    # two passes; the gating in a launch of its own
    (20000, 7, 5, 128), (300, 512, 16, 16), (1030, 1000, 4, 32)])
def test_gate_then_sort(tokens, experts, topk, block, dtype, masked):
    from flydsl_amd.kernels.moe.moe_sorting import moe_softmax_sort_flydsl, moe_sorting_flydsl, moe_sorting_get_workspace_size
    from flydsl_amd.kernels.moe.topk_gating_softmax import build_topk_gating_softmax_module

    g = torch.Generator(device="cuda").manual_seed(tokens + experts)
    logits = torch.randn(tokens, experts, generator=g, device="cuda").to(dtype)
    logits[1::3, : experts // 2] = 0.5  # ties
    logits[5] = float("nan")
    logits[7] = float("-inf")
    mask = (torch.rand(experts, generator=g, device="cuda") < 0.7).int() if masked else None
    name = "bf16" if dtype == torch.bfloat16 else "f32"
    ids, w = torch.empty(tokens, topk, dtype=torch.int32, device="cuda"), torch.empty(tokens, topk, device="cuda")
    build_topk_gating_softmax_module(experts, topk, name, True)(logits, w, ids, torch.empty_like(ids), tokens, stream=torch.cuda.current_stream())
    want = _outputs(tokens, topk, experts, block)
    moe_sorting_flydsl(ids, w, *want, None, experts, block, mask, workspace=False)
    size = moe_sorting_get_workspace_size(tokens, experts, topk)
    assert size > 0
    ws = torch.full((size,), 255, dtype=torch.uint8, device="cuda")
    ids2, w2, got = torch.empty_like(ids), torch.empty_like(w), _outputs(tokens, topk, experts, block)
    buf = torch.ones(1000, 16, dtype=torch.int32, device="cuda")
    moe_softmax_sort_flydsl(logits, *got, buf, experts, topk, name, block, mask, True, topk_ids=ids2, topk_weights=w2, workspace=ws, stream=torch.cuda.current_stream())
    assert torch.equal(ids, ids2) and torch.equal(w.view(torch.int32), w2.view(torch.int32)) and not buf.any()
    assert all(torch.equal(a.view(torch.int32), b.view(torch.int32)) for a, b in zip(got, want))


@pytest.mark.parametrize("masked", [False, True])
@pytest.mark.parametrize("tokens,experts,topk,block", [(4096, 32, 8, 128), (1500, 1024, 8, 32), (1500, 1025, 8, 32), (700, 3000, 7, 16), (33333, 5, 3, 64), (5000, 300, 1, 32)])
def test_sorter_with_and_without_slices(tokens, experts, topk, block, masked):
    from flydsl_amd.kernels.moe.moe_sorting import moe_sorting_flydsl, moe_sorting_get_workspace_size

    g = torch.Generator(device="cuda").manual_seed(tokens)
    ids = torch.randint(-1, experts + 1, (tokens, topk), generator=g, device="cuda", dtype=torch.int32)  # ids outside the range are dropped
    ids[: tokens // 3] = experts // 2  # most pairs to one expert
    w = torch.rand(tokens, topk, generator=g, device="cuda")
    mask = (torch.rand(experts, generator=g, device="cuda") < 0.5).int() if masked else None
    ws = torch.full((moe_sorting_get_workspace_size(tokens, experts, topk),), 255, dtype=torch.uint8, device="cuda")
    outs = []
    for workspace in (False, ws):
        outs.append(_outputs(tokens, topk, experts, block))
        moe_sorting_flydsl(ids, w, *outs[-1], None, experts, block, mask, workspace=workspace)
    assert all(torch.equal(a.view(torch.int32), b.view(torch.int32)) for a, b in zip(*outs))
