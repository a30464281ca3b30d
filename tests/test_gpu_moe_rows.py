"""Stage 2 of the MoE pairs accumulating by way of one row per sorted position, against a float64 restatement.  The operands are
small whole numbers (rows of zeros and ones against sparse weights of -1, 0, 1, all scales 1), so every sum of up to 256 in
magnitude is exact in bf16 and fp16 and the results must be equal, whatever the order of the additions.  The sorted lists hold
what the device has to find out by itself: tokens named more often than topk times, tokens without a row, padding ids in the
middle of a block, blocks whose expert does not exist, and blocks past the rows in use."""

import sys

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def _sorted_list(tokens, topk, experts, block, g):
    """Hand-made: (ids, expert of every block, rows in use)."""
    ids, eids = [], []
    for e in range(experts):
        n = int(torch.randint(0, 2 * block, (1,), generator=g))
        toks = torch.randint(0, max(1, tokens - 1), (n,), generator=g)  # repeats; the last token never occurs
        rows = [(int(torch.randint(0, topk, (1,), generator=g)) << 24) | int(t) for t in toks]
        if n > 3:
            rows[2] = tokens  # padding in the middle
        while len(rows) % block:
            rows.append(tokens | (topk << 24))
        ids += rows
        eids += [e if e != 1 else experts + 5] * (len(rows) // block)  # the blocks of expert 1 have no expert
    used = len(ids)
    ids += [0] * (2 * block)  # past the rows in use: looks like token 0
    eids += [0, 0]
    return ids, eids, used


@pytest.mark.parametrize("out_dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("kind,tokens,topk,block,model,inter", [
    ("mx", 1, 1, 16, 256, 256), ("mx", 37, 3, 32, 512, 256), ("mx", 300, 8, 64, 2304, 256), ("mx", 333, 9, 128, 4352, 512),
    ("fp8", 1, 1, 16, 64, 128), ("fp8", 37, 3, 32, 192, 128), ("int8", 300, 8, 64, 2112, 256), ("int8", 290, 5, 128, 4160, 384),
    ("fp8", 290, 8, 128, 4160, 512), ("int4", 61, 9, 128, 256, 256)])
def test_stage2_by_rows_equals_the_exact_sum(monkeypatch, kind, tokens, topk, block, model, inter, out_dtype):
    from flydsl_amd import _lib, layout
    from flydsl_amd.kernels.moe.moe_gemm_2stage import compile_moe_gemm2
    from flydsl_amd.kernels.moe.mxfp_moe import flydsl_mxfp4_gemm2

    experts = 4
    g = torch.Generator().manual_seed(tokens * 31 + block)
    ids, eids, used = _sorted_list(tokens, topk, experts, block, g)
    size = len(ids)
    dev = dict(device="cuda")
    sid, se = torch.tensor(ids, dtype=torch.int32, **dev), torch.tensor(eids, dtype=torch.int32, **dev)
    nv = torch.tensor([used, tokens], dtype=torch.int32, **dev)
    wts = torch.randint(1, 3, (size,), generator=g).float()
    w = (torch.rand(experts, model, inter, generator=g) < 8.0 / inter).int() * (torch.randint(0, 2, (experts, model, inter), generator=g) * 2 - 1)
    out0 = torch.randint(-4, 5, (tokens, model), generator=g).to(out_dtype)
    out = out0.cuda()
    calls = []

    def bytes_(t, k, s, dim, od, mx):
        calls.append(1)
        return s * dim * 2 + (t + 1) * 4 + t * k * 4 + s * 4 + 64

    monkeypatch.setattr(_lib.lib(), "psg_moe_rows_workspace_bytes", bytes_)
    rows = tokens * topk if kind != "mx" else size
    x = torch.randint(0, 2, (rows, inter), generator=g)
    if kind == "mx":
        code = lambda v: torch.where(v > 0, 2, torch.where(v < 0, 10, 0)).to(torch.uint8)
        pack = lambda v: (code(v[..., 0::2]) | (code(v[..., 1::2]) << 4)).contiguous()
        ones = lambda r: torch.full(((r + 31) // 32 * 32, inter // 32), 127, dtype=torch.uint8, **dev)
        flydsl_mxfp4_gemm2(inter_sorted_quant=pack(x).cuda(), inter_sorted_shuffled_scale=ones(size), w2_u8=layout.shuffle_weight_w4(pack(w).view(experts * model, -1)).cuda(),
                           w2_scale_u8=ones(experts * model), sorted_expert_ids=se, cumsum_tensor=nv, sorted_token_ids=sid, sorted_weights=wts.cuda(), flat_out=out,
                           M_logical=tokens, max_sorted=size, BM=block, epilog="atomic", NE=experts, D_HIDDEN=model, D_INTER=inter, topk=topk)
    else:
        td = torch.float8_e4m3fn if kind == "fp8" else torch.int8
        wq = w.view(experts * model, inter).to(td)
        ws = layout.shuffle_weight(wq.view(torch.int8))
        ws = layout.pack_shuffled_int8_to_int4(ws) if kind == "int4" else ws.view(td)
        fn = compile_moe_gemm2(model_dim=model, inter_dim=inter, experts=experts, topk=topk, tile_m=block, tile_n=64, tile_k=128, doweight_stage2=True,
                               out_dtype="bf16" if out_dtype == torch.bfloat16 else "f16", accumulate=True, in_dtype=kind)
        fn(out, x.to(td).cuda(), ws.contiguous().cuda(), torch.ones(rows, **dev), torch.ones(experts * model, **dev), sid, se, wts.cuda(), nv,
           tokens, model, inter, len(eids), torch.cuda.current_stream())
    torch.cuda.synchronize()
    assert calls, "the way by rows was not taken"
    want = out0.double()
    for blk, e in enumerate(eids):
        if blk * block >= used or e >= experts:
            continue
        pos = torch.arange(blk * block, (blk + 1) * block)
        t, s = torch.tensor(ids)[pos] & 0xFFFFFF, torch.tensor(ids)[pos] >> 24
        ok = (t < tokens) & ((s < topk) if kind != "mx" else torch.ones_like(t, dtype=torch.bool))
        src = pos[ok] if kind == "mx" else (t * topk + s)[ok]
        want.index_add_(0, t[ok], (x[src].double() @ w[e].double().T) * wts[pos[ok]].double()[:, None])
    assert want.abs().max() <= 256
    assert torch.equal(out.cpu().double(), want)


class _RealRule:
    """In place of monkeypatch above: the library's own rule and size, watched instead of replaced."""

    def __init__(self, monkeypatch):
        self.monkeypatch = monkeypatch

    def setattr(self, obj, name, seen):
        real = getattr(obj, name)

        def rule(*args):
            seen(*args)
            need = real(*args)
            assert need > 0, "the rule does not take this call by rows"
            return need

        self.monkeypatch.setattr(obj, name, rule)


@pytest.mark.parametrize("kind,tokens,topk,block,model,inter", [("mx", 410, 8, 64, 2048, 256), ("fp8", 515, 6, 128, 4096, 128), ("int8", 813, 4, 32, 4096, 128), ("int4", 410, 8, 64, 4096, 128)])
def test_stage2_by_rows_where_the_library_takes_it(monkeypatch, kind, tokens, topk, block, model, inter):
    test_stage2_by_rows_equals_the_exact_sum(_RealRule(monkeypatch), kind, tokens, topk, block, model, inter, torch.bfloat16)


def _full_list(tokens, topk, experts, block, g):
    """The list a sorter makes: every (token, slot) once, each expert's rows filled up to whole blocks."""
    expert = torch.randint(0, experts, (tokens, topk), generator=g)
    ids, eids = [], []
    for e in range(experts):
        rows = [(s << 24) | t for t, s in (expert == e).nonzero().tolist()]
        rows += [tokens | (topk << 24)] * (-len(rows) % block)
        ids += rows
        eids += [e] * (len(rows) // block)
    return ids, eids, len(ids)


@pytest.mark.parametrize("kind,tokens,topk,block,model,inter", [
    ("int4", 830, 8, 64, 2048, 256), ("int4", 830, 8, 128, 2048, 384), ("int8", 830, 8, 64, 2048, 384), ("fp8", 830, 8, 64, 2048, 256), ("fp8", 515, 6, 32, 4096, 128),
    ("int8", 515, 6, 128, 4096, 128)])
def test_stage2_by_rows_of_a_whole_layer(monkeypatch, kind, tokens, topk, block, model, inter):
    """What an accumulating layer runs: all pairs in the list, more than two workgroups a CU on 128-column tiles."""
    monkeypatch.setattr(sys.modules[__name__], "_sorted_list", _full_list)
    test_stage2_by_rows_equals_the_exact_sum(_RealRule(monkeypatch), kind, tokens, topk, block, model, inter, torch.bfloat16)


@pytest.mark.parametrize("kind,tokens,topk,block,model,inter,rows", [
    ("int8", 9001, 3, 16, 64, 128, 50000), ("int4", 12347, 5, 32, 192, 128, 50000), ("fp8", 30011, 2, 64, 64, 128, 120000), ("fp8", 9001, 6, 128, 256, 256, 56000), ("mx", 9001, 3, 64, 256, 256, 130000)])
def test_long_lists(monkeypatch, kind, tokens, topk, block, model, inter, rows):
    """Lists that are made in launches of their own, by all CUs, and the longest the MX pair makes beside its tiles: more rows of some tokens than topk, tokens without one."""

    def long_list(tokens, topk, experts, block, g):
        ids, eids = [], []
        for e in range(experts):
            n = rows // experts + int(torch.randint(1, 2 * block, (1,), generator=g))
            t = torch.randint(0, tokens - 1, (n,), generator=g)
            t[:97 * 12:97] = t[0]  # (a dozen times from each of three experts: at most 36 rows of one token, whose sum stays below 256)
            t[::101] = tokens  # padding
            if e != 1:
                t[5::7] = t[5]
                t[5::7][2:] = tokens
            s = torch.randint(0, topk, (n,), generator=g)
            blk = torch.where(t == tokens, t, (s << 24) | t).tolist()
            blk += [tokens | (topk << 24)] * (-len(blk) % block)
            ids += blk
            eids += [e if e != 1 else experts + 5] * (len(blk) // block)
        return np.array(ids + [0] * block), eids + [0], len(ids)  # (an array: the comparison makes a tensor of it for every block)

    monkeypatch.setattr(sys.modules[__name__], "_sorted_list", long_list)
    test_stage2_by_rows_equals_the_exact_sum(monkeypatch, kind, tokens, topk, block, model, inter, torch.bfloat16)
