"""The 256-row tiles of the MoE stages against the 128-row kernel: the same sums in the same order, so the same bits.  The lists
are hand-made: runs of one, two, three and many blocks of an expert, runs cut up so that there are more tiles than a grouped list
of that length can have, more than 512 blocks, blocks without an expert, and blocks past the rows in use; the widths leave the last
column tile partly filled, the K extents cover one step up to more than the pipeline holds."""

import pytest
import torch

pytestmark = pytest.mark.gpu


def _launch(stage, kind, out_dtype, x, w, sx, sw, ids, eids, wts, used, tokens, topk, experts, n_out, K, pairing):
    from flydsl_amd.kernels.moe.moe_gemm_2stage import MoeStage

    model, inter = (K, n_out) if stage == 1 else (n_out, K)
    fn = MoeStage(stage, model, inter, experts, topk, 128, True, "bf16" if out_dtype == torch.bfloat16 else "f16", False, kind)
    fn.no_pairing = not pairing
    out = torch.zeros(tokens * topk, n_out, dtype=out_dtype, device="cuda")
    fn(out, x, w, sx, sw, ids, eids, wts, torch.tensor([used, tokens], dtype=torch.int32, device="cuda"), tokens, n_out, K, eids.numel(), torch.cuda.current_stream())
    torch.cuda.synchronize()
    return out


@pytest.mark.parametrize("kind,stage,n_out,K,runs,out_dtype", [
    ("fp8", 1, 2960, 128, [3, 1, 2, 7, 3], torch.bfloat16),
    ("fp8", 2, 5904, 640, [3, 1, 2, 7, 3], torch.float16),
    ("int8", 1, 3072, 896, [8, 5, 4], torch.float16),
    ("int8", 2, 6144, 1152, [2, 2, 9, 3], torch.bfloat16),
    ("fp8", 2, 2816, 256, [1] * 40, torch.bfloat16),        # every run odd: the grid's bound is exceeded, workgroups take a second tile
    ("fp8", 1, 1920, 256, [301, 230, 9], torch.bfloat16),    # 540 blocks
])
def test_same_bits_as_the_128_row_kernel(kind, stage, n_out, K, runs, out_dtype):
    g = torch.Generator(device="cuda").manual_seed(n_out + K)
    dev = dict(device="cuda")
    experts = 4
    blocks = sum(runs)
    tokens, topk = blocks * 128 // 2 + 3, 2  # enough rows per expert for the 256-row tiles
    eids = []
    for i, n in enumerate(runs):
        eids += [i % experts if i != 3 else experts + 1] * n  # run 3 has no expert
    used = (blocks - 1) * 128  # the last block is past the rows in use
    perm = torch.randperm(tokens * topk, generator=g, **dev)[: blocks * 128]
    ids = ((perm % topk) << 24 | (perm // topk)).int()
    ids[5::131] = tokens  # padding
    eids = torch.tensor(eids, dtype=torch.int32, **dev)
    wts = torch.rand(ids.numel(), generator=g, **dev)
    rows_x, rows_w = tokens * (1 if stage == 1 else topk), experts * n_out * (2 if stage == 1 else 1)
    td = torch.float8_e4m3fn if kind == "fp8" else torch.int8
    q = lambda r: (torch.randn(r, K, generator=g, **dev).mul_(20)).clamp_(-120, 120).to(td)
    args = (q(rows_x), q(rows_w), torch.rand(rows_x, generator=g, **dev), torch.rand(rows_w, generator=g, **dev) * 1e-3, ids, eids, wts, used, tokens, topk, experts, n_out, K)
    a = _launch(stage, kind, out_dtype, *args, pairing=True)
    b = _launch(stage, kind, out_dtype, *args, pairing=False)
    assert b.abs().sum() > 0
    assert torch.equal(a.view(torch.int16), b.view(torch.int16))
