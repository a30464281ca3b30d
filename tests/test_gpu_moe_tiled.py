"""The 128x256 tiles of the MoE stages on blocks of 128 rows against the kernel of the smaller tiles: the same sums in the same order, so the same bits.  The lists
are hand-made: runs of one, two, three and many blocks of an expert, more than 512 blocks, blocks without an expert, and blocks past the rows in use; the widths leave the last
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
    ("fp8", 2, 2816, 256, [1] * 40, torch.bfloat16),        # another expert for every block
    ("fp8", 1, 1920, 256, [301, 230, 9], torch.bfloat16),    # 540 blocks
])
def test_same_bits_as_the_smaller_tiles(kind, stage, n_out, K, runs, out_dtype):
    g = torch.Generator(device="cuda").manual_seed(n_out + K)
    dev = dict(device="cuda")
    experts = 4
    blocks = sum(runs)
    tokens, topk = blocks * 128 // 2 + 3, 2  # enough rows per expert for the 128x256 tiles
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


def _blocks(runs, experts):
    eids = []
    for i, n in enumerate(runs):
        eids += [i % experts if i != 3 else experts + 1] * n  # run 3 has no expert
    return eids


@pytest.mark.parametrize("kind,n_out,K,runs,out_dtype", [
    ("fp8", 5904, 640, [3, 1, 2, 7, 3], torch.float16), ("int8", 6144, 1152, [2, 2, 9, 3], torch.bfloat16), ("fp8", 2816, 256, [1] * 40, torch.bfloat16)])
def test_atomic_epilogue_equals_the_exact_sum(kind, n_out, K, runs, out_dtype):
    """Accumulating without scratch (two slots: added directly): small whole numbers, exact in 16 bits whatever the order of the additions."""
    from flydsl_amd import layout
    from flydsl_amd.kernels.moe.moe_gemm_2stage import MoeStage

    g = torch.Generator(device="cuda").manual_seed(n_out + K)
    dev = dict(device="cuda")
    experts, topk = 4, 2
    eids = _blocks(runs, experts)
    blocks = len(eids)
    tokens, used = blocks * 64 + 3, (blocks - 1) * 128
    perm = torch.randperm(tokens * topk, generator=g, **dev)[: blocks * 128]
    ids = ((perm % topk) << 24 | (perm // topk)).int()
    ids[5::131] = tokens  # padding
    wts = torch.randint(1, 3, (blocks * 128,), generator=g, **dev).float()
    x = torch.randint(0, 2, (tokens * topk, K), generator=g, **dev).float()
    w = (torch.rand(experts * n_out, K, generator=g, **dev) < 8.0 / K).float() * (torch.randint(0, 2, (experts * n_out, K), generator=g, **dev) * 2 - 1)
    td = torch.float8_e4m3fn if kind == "fp8" else torch.int8
    out0 = torch.randint(-4, 5, (tokens, n_out), generator=g, **dev).to(out_dtype)
    out = out0.clone()
    fn = MoeStage(2, n_out, K, experts, topk, 128, True, "bf16" if out_dtype == torch.bfloat16 else "f16", True, kind)
    fn(out, x.to(td), layout.shuffle_weight(w.to(td).view(torch.int8)).view(td).contiguous(), torch.ones(tokens * topk, **dev), torch.ones(experts * n_out, **dev), ids,
       torch.tensor(eids, dtype=torch.int32, **dev), wts, torch.tensor([used, tokens], dtype=torch.int32, **dev), tokens, n_out, K, blocks, torch.cuda.current_stream())
    want = out0.float()
    for blk, e in enumerate(eids):
        if blk * 128 >= used or e >= experts:
            continue
        rows = slice(blk * 128, (blk + 1) * 128)
        t, s = (ids[rows] & 0xFFFFFF).long(), (ids[rows] >> 24).long()
        ok = t < tokens
        # fp32 products of whole numbers: exact
        want.index_add_(0, t[ok], (x[(t * topk + s)[ok]] @ w[e * n_out:(e + 1) * n_out].T) * wts[rows][ok][:, None])
    assert want.abs().max() <= 256 and not torch.equal(want, out0.float())
    assert torch.equal(out.float(), want)


def test_slot_major_activations():
    """Stage 1 of "int8smooth" reads one row of x per (slot, token) at slot * tokens + token."""
    g = torch.Generator(device="cuda").manual_seed(5)
    dev = dict(device="cuda")
    experts, topk, n_out, K = 4, 2, 3072, 896
    eids = _blocks([8, 5, 4], experts)
    blocks = len(eids)
    tokens = blocks * 64 + 3
    perm = torch.randperm(tokens * topk, generator=g, **dev)[: blocks * 128]
    ids = ((perm % topk) << 24 | (perm // topk)).int()
    ids[5::131] = tokens
    q = lambda r: torch.randint(-120, 121, (r, K), generator=g, dtype=torch.int8, **dev)
    args = (q(tokens * topk), q(experts * 2 * n_out), torch.rand(tokens * topk, generator=g, **dev), torch.rand(experts * 2 * n_out, generator=g, **dev) * 1e-3, ids,
            torch.tensor(eids, dtype=torch.int32, **dev), torch.rand(blocks * 128, generator=g, **dev), blocks * 128, tokens, topk, experts, n_out, K)
    a, b = (_launch(1, "int8smooth", torch.bfloat16, *args, pairing=p) for p in (True, False))
    # the rows are those of the slot: other rows for the second slot give other results there, and there only
    other = list(args)
    other[0] = torch.cat([args[0][:tokens], q(tokens)])
    c = _launch(1, "int8smooth", torch.bfloat16, *other, pairing=True)
    assert b.abs().sum() > 0
    assert torch.equal(a.view(torch.int16), b.view(torch.int16))
    changed = (c != a).any(1).view(tokens, topk)
    assert not changed[:, 0].any() and changed[:, 1].any()
