"""The builds of the MoE stages that ask for their operands one and three steps ahead, on both sides of the rule that chooses them and on every remainder of
the K steps by the four register sets; blocks of 16 and 32 rows with weights read past the caches (more than these hold) and, from three workgroups a CU on, two blocks of 16 rows of an
expert at a time in every stage, through the caches and past them.  Whole numbers as operands and powers of two as scales: the sums are exact, stage 2 is one rounding of them."""

import pytest
import torch

pytestmark = pytest.mark.gpu

SHAPES = [(64, 130, 2, 4, 64), (128, 300, 3, 4, 192), (128, 290, 1, 2, 128), (64, 700, 2, 4, 4096), (128, 900, 2, 4, 4160), (32, 130, 2, 4, 192),
          (16, 40, 2, 4, 192), (16, 12, 3, 8, 128)]
# Two blocks of 16 rows a workgroup, rows an expert: 12.5 stage 1 of one-byte weights and every stage 2, 15 stage 1 of int4 weights too, at most 24 past the caches where the
# weights are more than these hold (stage 1 and 2, fp8: from 8 steps on; int4: from 9, an odd number of which stage 1 doubles), 25 through them
PAIRED = [(16, 200, 2, 32, 4096), (16, 240, 2, 32, 4096), (16, 400, 2, 32, 4096)]
STREAMED = [(16, 20, 2, 32, 4160, 13), (16, 20, 2, 32, 4160, 14), (16, 20, 2, 32, 4160, 15), (16, 20, 2, 32, 4160, 16), (32, 60, 2, 32, 4160, 14), (32, 60, 2, 32, 4160, 15)]


@pytest.mark.parametrize("kind", ["fp8", "int8", "int4"])
@pytest.mark.parametrize("block,tokens,topk,experts,n_out,steps", [s + (k,) for s in SHAPES for k in (1, 2, 3, 4, 5, 6, 7, 8, 11) if s[4] < 4000 or k <= 4]
                         + STREAMED + [s + (k,) for s in PAIRED for k in (8, 9, 10, 11)])
@pytest.mark.parametrize("stage", [1, 2])
def test_depths(stage, block, tokens, topk, experts, n_out, kind, steps):
    from flydsl_amd import layout
    from flydsl_amd.kernels.moe.moe_gemm_2stage import compile_moe_gemm1, compile_moe_gemm2
    from flydsl_amd.kernels.moe.moe_sorting import moe_sorting

    K = 128 * steps
    if stage == 1 and steps % 2:
        K *= 2  # the builder wants an even number of steps there
    g = torch.Generator(device="cuda").manual_seed(steps + block)
    logits = torch.randn(tokens, experts, generator=g, device="cuda")
    wts, ids = logits.softmax(-1).topk(topk, dim=-1)
    wts = 2.0 ** torch.randint(-2, 2, wts.shape, generator=g, device="cuda").float()
    sid, swt, se, nv = moe_sorting(ids.int(), wts, num_experts=experts, block_size=block)
    rows_x, rows_w = (tokens, 2 * n_out) if stage == 1 else (tokens * topk, n_out)
    x, w = (torch.randint(-4, 5, (r, K), generator=g, device="cuda") for r in (rows_x, experts * rows_w))
    td = torch.float8_e4m3fn if kind == "fp8" else torch.int8
    ws = layout.shuffle_weight(w.to(td).view(torch.int8))
    ws = layout.pack_shuffled_int8_to_int4(ws) if kind == "int4" else ws.view(td)
    sx, sw = (2.0 ** torch.randint(-9, -5, (r,), generator=g, device="cuda").float() for r in (rows_x, experts * rows_w))
    kw = dict(experts=experts, topk=topk, tile_m=block, tile_n=64, tile_k=128, in_dtype=kind, out_dtype="bf16")
    if stage == 1:
        fn = compile_moe_gemm1(model_dim=K, inter_dim=n_out, doweight_stage1=False, **kw)
    else:
        fn = compile_moe_gemm2(model_dim=n_out, inter_dim=K, doweight_stage2=True, accumulate=False, **kw)
    out = torch.full((tokens * topk, n_out), -8192.0, dtype=torch.bfloat16, device="cuda")
    fn(out, x.to(td), ws.contiguous(), sx, sw, sid, se, swt, nv, tokens, n_out, K, se.numel(), torch.cuda.current_stream())
    xs = (x.double() * sx.double()[:, None]).view(rows_x, K)
    wsd = (w.double() * sw.double()[:, None]).view(experts, rows_w, K)
    want = torch.empty(tokens, topk, n_out, dtype=torch.float64, device="cuda")
    for e in range(experts):
        t, s = (ids == e).nonzero(as_tuple=True)
        y = (xs[t] if stage == 1 else xs[t * topk + s]) @ wsd[e].T
        if stage == 1:
            gate, up = y[:, :n_out], y[:, n_out:]
            y = gate / (1 + torch.exp(-gate)) * up
        want[t, s] = y
    want = want.view(tokens * topk, n_out)
    if stage == 2:
        assert torch.equal(out, (want * wts.view(-1, 1).double()).float().bfloat16())
    else:
        # half a unit in the last place of bf16, and the fp32 exponential and division
        assert ((out.double() - want).abs() <= (2.0 ** -8 + 2.0 ** -18) * want.abs() + 1e-30).all()


@pytest.mark.parametrize("per_tile", [1, 2])
@pytest.mark.parametrize("runs,unused", [([1] * 20, 0), ([1] * 20, 1), ([3, 1, 2, 1, 4], 0), ([3, 1, 2, 1, 4], 2), ([1] * 64, 0), ([1] * 65, 0), ([2] * 64, 0), ([1, 2] * 43, 0), ([1, 2] * 43, 3),
                                         ([1] * 300, 0), ([5] + [1] * 200 + [64, 1, 1], 0), ([7], 0), ([2, 2], 4)])
def test_the_only_tile_of_an_expert_reads_past_the_caches(runs, unused, per_tile):
    """... and only where more experts have rows than the caches hold: over runs of blocks, some without an expert, the last ones not in use."""
    from flydsl_amd import _lib

    experts, handle = len(runs) + 5, _lib.lib()
    ids = [e if e % 7 != 3 else (-1 if e % 2 else experts + 2) for e, n in enumerate(runs) for _ in range(n)]
    used = len(ids) - unused
    seen = len({e for e in ids[:used] if 0 <= e < experts})
    t = torch.tensor(ids, dtype=torch.int32, device="cuda")
    for cached in (0, max(seen - 1, 0), seen):
        want = []
        for i, e in enumerate(ids):
            alone = (i == 0 or ids[i - 1] != e) and not (i + per_tile < used and ids[i + per_tile] == e)
            want.append(-1 if i >= used or not 0 <= e < experts else int(alone and seen > cached))
        out = torch.full((len(ids),), -5, dtype=torch.int32, device="cuda")
        rc = handle.psg_debug_moe_reads_once(t.data_ptr(), len(ids), used, per_tile, experts, cached, out.data_ptr(), _lib.stream_handle(None))
        assert rc == 0, handle.psg_last_error()
        assert out.tolist() == want, cached
