"""The native launch path accepts what the checks in Python accept and leaves everything else to them: same results, same errors."""

import pytest
import torch

from flydsl_amd import _lib

pytestmark = pytest.mark.gpu


@pytest.fixture
def rcs(monkeypatch):
    """Return codes of the native calls, as they come."""
    seen = []

    class Watched:
        DECLINED = _lib._native.DECLINED

        def __getattr__(self, name):
            fn = getattr(real, name)
            return lambda *a: seen.append(fn(*a)) or seen[-1]

    real = _lib._native
    monkeypatch.setattr(_lib, "_native", Watched())
    return seen


def _mx(M=33, N=64, K=256, batch=1):
    g = torch.Generator(device="cuda").manual_seed(1)
    byte = lambda n: torch.randint(0, 256, (n,), generator=g, device="cuda", dtype=torch.uint8)
    scale = lambda n: torch.randint(126, 129, (n,), generator=g, device="cuda", dtype=torch.uint8)
    return dict(c=torch.zeros(batch, M, N, dtype=torch.bfloat16, device="cuda"), a=byte(batch * M * K // 2), b=byte(batch * N * K // 2),
                sa=scale(batch * ((M + 31) // 32 * 32) * (K // 32)), sb=scale(batch * N * (K // 32)), M=M, N=N, K=K)


def _launch(d, stream, **kw):
    from kernels.gemm.mxfp4_preshuffle import launch_gemm

    o = dict(d, **kw)
    launch_gemm(o["c"], o["a"], o["b"], o["sa"], o["sb"], o["M"], o["N"], stream, o["N"], o["K"], 64, 128, 256, "fp4", "bf16", "fp4", 1, -1, -1, -1, -1, -1, -1, 0, 0)
    return o["c"]


def test_mx_launch_and_what_it_declines(rcs):
    s = torch.cuda.current_stream()
    d = _mx()
    want = _launch(d, s).clone()
    assert rcs == [0] and want.count_nonzero() > 0
    declined = _lib._native.DECLINED
    # raw addresses, a stream given as nothing: the Python path, same bits
    d["c"].zero_()
    assert torch.equal(_launch(d, s, a=d["a"].data_ptr()), want) and rcs[-1] == declined
    assert torch.equal(_launch(d, None), want) and len(rcs) == 2
    assert torch.equal(_launch(d, s.cuda_stream), want) and rcs[-1] == 0
    for bad in (dict(a=d["a"][:-1]), dict(c=d["c"][:, :-1].contiguous()), dict(b=d["b"].cpu()), dict(sa=d["sa"].view(-1, 2)[:, 0])):
        with pytest.raises(ValueError):
            _launch(d, s, **bad)
        assert rcs[-1] == declined
    with pytest.raises(ValueError, match="aligned"):  # refused by the library itself
        _launch(d, s, a=torch.zeros(d["a"].numel() + 1, dtype=torch.uint8, device="cuda")[1:])
    assert rcs[-1] < 0 and rcs[-1] != declined


def test_quantisers(rcs):
    from flydsl_amd import quant_device as Q

    s, declined = torch.cuda.current_stream(), _lib._native.DECLINED
    x = torch.randn(33, 512, device="cuda", dtype=torch.bfloat16)
    y, sc = torch.empty(33, 512, dtype=torch.int8, device="cuda"), torch.empty(33, device="cuda")
    got = Q.pertoken_quant(x, torch.int8, stream=s, out=(y, sc))
    assert rcs == [0] and got[0] is y and got[1].shape == (33, 1)
    want = Q.pertoken_quant(x, torch.int8)
    assert torch.equal(got[0], want[0]) and torch.equal(got[1], want[1])
    p, e = torch.empty(33, 256, dtype=torch.uint8, device="cuda"), torch.empty(64, 16, dtype=torch.uint8, device="cuda")
    got = Q.per_1x32_f4_quant(x, shuffle=True, stream=s, out=(p, e))
    want = Q.per_1x32_f4_quant(x, shuffle=True)
    assert rcs[-1] == 0 and all(torch.equal(a.view(torch.uint8), b.view(torch.uint8)) for a, b in zip(got, want))
    for fn, bad in ((lambda o: Q.pertoken_quant(x, torch.int8, stream=s, out=o), [(y[:32], sc), (y, sc[:32]), (y, sc.half()), (y.t(), sc), (y.cpu(), sc)]),
                    (lambda o: Q.per_1x32_f4_quant(x, stream=s, out=o), [(p[:32], e), (p, e[:32]), (p.t(), e)])):
        for o in bad:
            with pytest.raises(ValueError):
                fn(o)
            assert rcs[-1] == declined
    with pytest.raises(TypeError):
        Q.pertoken_quant(x.double(), torch.int8, stream=s, out=(y, sc))
    with pytest.raises(ValueError):
        Q.pertoken_quant(x[:, :500], torch.int8, stream=s, out=(y, sc))


@pytest.mark.parametrize("tokens", [5, 700])  # one launch, and gating and sorting one after the other
def test_routing(rcs, tokens):
    from flydsl_amd.kernels.moe.moe_sorting import moe_softmax_sort_flydsl, sorted_sizes

    s, declined, E, topk, B = torch.cuda.current_stream(), _lib._native.DECLINED, 16, 4, 32
    logits = torch.randn(tokens, E, device="cuda", dtype=torch.bfloat16)
    rows, blocks = sorted_sizes(tokens, topk, E, B)

    def go(stream=s, **kw):
        o = dict(sid=torch.empty(rows, dtype=torch.int32, device="cuda"), sw=torch.empty(rows, device="cuda"), se=torch.empty(blocks, dtype=torch.int32, device="cuda"),
                 nv=torch.empty(2, dtype=torch.int32, device="cuda"), buf=torch.ones(tokens, 64, dtype=torch.bfloat16, device="cuda"),
                 ids=torch.empty(tokens, topk, dtype=torch.int32, device="cuda"), w=torch.empty(tokens, topk, device="cuda"))
        o.update(kw)
        moe_softmax_sort_flydsl(logits, o["sid"], o["sw"], o["se"], o["nv"], o["buf"], E, topk, "bf16", B, None, True, None, topk_ids=o["ids"], topk_weights=o["w"], stream=stream)
        return o

    want, n = go(stream=None), len(rcs)
    got = go()
    assert n == 0 and rcs == [0] and not got["buf"].any()
    assert all(torch.equal(got[k], want[k]) for k in want)
    if tokens == 5:  # the routing itself is an extra there
        more = go(ids=None, w=None)
        assert rcs[-1] == 0 and torch.equal(more["sid"], want["sid"])
    for bad in (dict(sid=want["sid"][:-1]), dict(sw=want["sw"].half()), dict(se=want["se"][:-1]), dict(nv=want["nv"][:1]), dict(w=want["w"].int()), dict(ids=want["ids"][:-1])):
        with pytest.raises(ValueError):
            go(**bad)
        assert rcs[-1] == declined


@pytest.mark.parametrize("stage", [1, 2])
def test_moe_stages(rcs, stage):
    from flydsl_amd.kernels.moe.moe_gemm_2stage import compile_moe_gemm1, compile_moe_gemm2, compile_moe_reduction

    s, declined, E, topk, tokens, model, inter = torch.cuda.current_stream(), _lib._native.DECLINED, 2, 2, 3, 256, 128
    kw = dict(model_dim=model, inter_dim=inter, experts=E, topk=topk, tile_m=16, tile_n=64, tile_k=128, out_dtype="bf16", in_dtype="int8")
    fn = compile_moe_gemm1(doweight_stage1=False, **kw) if stage == 1 else compile_moe_gemm2(doweight_stage2=True, accumulate=False, **kw)
    g = torch.Generator(device="cuda").manual_seed(3)
    K, n, rows_x = (model, inter, tokens) if stage == 1 else (inter, model, tokens * topk)
    i8 = lambda *sh: torch.randint(-8, 9, sh, generator=g, device="cuda", dtype=torch.int8)
    ids = torch.full((32,), tokens, dtype=torch.int32, device="cuda")
    for i, (t, k) in enumerate([(0, 0), (1, 0), (2, 1)]):
        ids[i], ids[16 + i] = t | (k << 24), t | ((1 - k) << 24)
    a = dict(out=torch.zeros(tokens * topk, n, dtype=torch.bfloat16, device="cuda"), x=i8(rows_x, K), w=i8(E * (2 * n if stage == 1 else n), K), sx=torch.ones(rows_x, device="cuda"),
             sw=torch.full((E * (2 * n if stage == 1 else n),), 0.01, device="cuda"), ids=ids, se=torch.tensor([0, 1], dtype=torch.int32, device="cuda"),
             swt=torch.ones(32, device="cuda"), nv=torch.tensor([32, tokens], dtype=torch.int32, device="cuda"))

    def go(stream=s, **over):
        o = dict(a, **over)
        fn(*o.values(), tokens, n, K, 2, stream)
        return o["out"].clone()

    want = go(stream=None)
    assert want.count_nonzero() and not rcs
    a["out"].zero_()
    assert torch.equal(go(), want) and rcs == [0]
    bad = [dict(out=a["out"][:-1]), dict(x=a["x"][:-1]), dict(w=a["w"][:-1]), dict(sx=a["sx"][:-1]), dict(sw=a["sw"].half()), dict(se=a["se"][:1]), dict(nv=a["nv"].cpu()), dict(swt=None)]
    for b in bad:
        with pytest.raises(ValueError):
            go(**b)
        assert rcs[-1] == declined
    if stage == 2:
        red = compile_moe_reduction(topk=topk, model_dim=model, dtype_str="bf16")
        y = torch.empty(tokens, model, dtype=torch.bfloat16, device="cuda")
        red(want, y, None, None, tokens, s)
        assert rcs[-1] == 0 and torch.equal(y, want.view(tokens, topk, model).float().sum(1).bfloat16())
        with pytest.raises(ValueError):
            red(want[:-1], y, None, None, tokens, s)
        assert rcs[-1] == declined


def test_fused_mx_pair(rcs):
    from flydsl_amd.kernels.moe.mxfp_moe import flydsl_mxfp4_gemm1, flydsl_mxfp4_gemm2, moe_mxfp4_sort

    s, declined, E, tokens, H, I = torch.cuda.current_stream(), _lib._native.DECLINED, 2, 3, 256, 256
    g = torch.Generator(device="cuda").manual_seed(5)
    byte = lambda *sh: torch.randint(0, 256, sh, generator=g, device="cuda", dtype=torch.uint8)
    one = lambda *sh: torch.full(sh, 124, dtype=torch.uint8, device="cuda")
    ids = torch.full((64,), tokens, dtype=torch.int32, device="cuda")
    ids[:2], ids[32] = torch.tensor([0, 2], dtype=torch.int32), 1
    se, nv = torch.tensor([0, 1], dtype=torch.int32, device="cuda"), torch.tensor([64, tokens], dtype=torch.int32, device="cuda")
    scales = one(tokens, H // 32)
    sort = lambda stream, out, **kw: moe_mxfp4_sort(kw.get("scales", scales), ids, nv, tokens, block_size=32, out=out, stream=stream)
    xs = [sort(st, byte(64, H // 32)) for st in (None, s)]
    assert rcs == [0] and torch.equal(*xs)
    k1 = dict(a_quant=byte(tokens, H // 2), a_scale_sorted_shuffled=xs[0], w1_u8=byte(E * 2 * I, H // 2), w1_scale_u8=one(E * 2 * I, H // 32), sorted_expert_ids=se, cumsum_tensor=nv,
              m_indices=ids, n_tokens=tokens, BM=32, NE=E, D_HIDDEN=H, D_INTER=I, topk=1)
    first = lambda stream, **kw: flydsl_mxfp4_gemm1(**{**k1, **dict(inter_sorted_quant=torch.zeros(64, I // 2, dtype=torch.uint8, device="cuda"),
                                                                   inter_sorted_shuffled_scale=torch.zeros(64, I // 32, dtype=torch.uint8, device="cuda")), **kw}, stream=stream)
    h = [first(st) for st in (None, s)]
    assert rcs[-1] == 0 and all(torch.equal(p, q) for p, q in zip(*h)) and h[0][0].count_nonzero()
    k2 = dict(inter_sorted_quant=h[0][0], inter_sorted_shuffled_scale=h[0][1], w2_u8=byte(E * H, I // 2), w2_scale_u8=one(E * H, I // 32), sorted_expert_ids=se, cumsum_tensor=nv,
              sorted_token_ids=ids, sorted_weights=torch.ones(64, device="cuda"), M_logical=tokens, max_sorted=64, BM=32, epilog="atomic", NE=E, D_HIDDEN=H, D_INTER=I, topk=1)
    second = lambda stream, **kw: flydsl_mxfp4_gemm2(**{**k2, "flat_out": torch.zeros(tokens, H, dtype=torch.bfloat16, device="cuda"), **kw}, stream=stream)
    y = [second(st) for st in (None, s)]
    assert rcs[-1] == 0 and torch.equal(*y) and y[0].count_nonzero()
    n = len(rcs)
    for call, bad in ((first, dict(w1_u8=k1["w1_u8"][:-1])), (first, dict(m_indices=ids.long())), (first, dict(a_quant=k1["a_quant"][:-1])), (first, dict(a_scale_sorted_shuffled=None)),
                      (second, dict(sorted_weights=k2["sorted_weights"].half())), (second, dict(flat_out=torch.zeros(tokens - 1, H, dtype=torch.bfloat16, device="cuda"))),
                      (second, dict(w2_scale_u8=k2["w2_scale_u8"][:-1]))):
        with pytest.raises((ValueError, TypeError)):
            call(s, **bad)
    assert rcs[n:] == [declined] * 7
    with pytest.raises(NotImplementedError):
        first(s, interleave=True)
    with pytest.raises(NotImplementedError):
        second(s, BM=48)


def test_tensors_without_an_address_are_refused_with_an_error(rcs):
    """Under vmap a tensor looks like a plain device tensor and has no storage: asking for its address throws in native code."""
    from flydsl_amd import quant_device as Q
    from flydsl_amd.kernels.moe.moe_gemm_2stage import compile_moe_reduction
    from flydsl_amd.kernels.moe.mxfp_moe import moe_mxfp4_sort

    s, declined = torch.cuda.current_stream(), _lib._native.DECLINED
    dev = dict(device="cuda")
    x = torch.randn(2, 32, 256, dtype=torch.bfloat16, **dev)
    y, sc = torch.empty(32, 256, dtype=torch.int8, **dev), torch.empty(32, **dev)
    p, e = torch.empty(32, 128, dtype=torch.uint8, **dev), torch.empty(32, 8, dtype=torch.uint8, **dev)
    red, r = compile_moe_reduction(topk=2, model_dim=64, dtype_str="bf16"), torch.empty(64, 64, dtype=torch.bfloat16, **dev)
    ids, nv = torch.zeros(32, dtype=torch.int32, **dev), torch.tensor([32, 32], dtype=torch.int32, **dev)
    scales = torch.ones(2, 32, 8, dtype=torch.uint8, **dev)
    for call, arg in ((lambda t: Q.pertoken_quant(t, torch.int8, stream=s, out=(y, sc)), x), (lambda t: Q.per_1x32_f4_quant(t, stream=s, out=(p, e)), x),
                      (lambda t: red(t, r, None, None, 64, s), x), (lambda t: moe_mxfp4_sort(t, ids, nv, 32, block_size=32, out=e, stream=s), scales)):
        n = len(rcs)
        with pytest.raises(RuntimeError):
            torch.func.vmap(call)(arg)
        assert rcs[n:] == [declined]


def test_without_the_extension_the_results_are_the_same(monkeypatch):
    from flydsl_amd import quant_device as Q

    s, d = torch.cuda.current_stream(), _mx()
    x, y, sc = torch.randn(33, 512, device="cuda"), torch.empty(33, 512, dtype=torch.int8, device="cuda"), torch.empty(33, device="cuda")
    go = lambda: [t.clone() for t in (_launch(d, s), *Q.pertoken_quant(x, torch.int8, stream=s, out=(y, sc)))]
    want = go()
    for t in (d["c"], y, sc):
        t.zero_()
    monkeypatch.setattr(_lib, "_native", _lib._Declines)
    assert all(torch.equal(a, b) for a, b in zip(go(), want))
