"""The second pass of the split-K plan with every number of slices that has a build of its own and one that has none, with and without scales, bias and activation, both output types.

Operands are whole numbers and scales and biases such that every sum and product is exact in fp32, so the result has one right value."""

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind,out,epi", [("int8", "bf16", "none"), ("fp8", "fp16", "bias"), ("bf16", "bf16", "bias_relu"), ("fp16", "fp16", "none")])
@pytest.mark.parametrize("splits", [2, 3, 4, 5, 6, 7, 8, 9])
def test_slices(kind, out, epi, splits):
    from flydsl_amd import layout
    from flydsl_amd.kernels.gemm.preshuffle_gemm import compile_preshuffle_gemm

    M, N, K = 37, 208, 64 * (2 * splits + 1)
    td = {"int8": torch.int8, "fp8": torch.float8_e4m3fn, "fp16": torch.float16, "bf16": torch.bfloat16}[kind]
    od = {"bf16": torch.bfloat16, "fp16": torch.float16}[out]
    scaled = kind in ("int8", "fp8")
    g = torch.Generator(device="cuda").manual_seed(splits)
    a, w = (torch.randint(-2, 3, (r, K), generator=g, device="cuda") for r in (M, N))
    sa, sb = (2.0 ** torch.randint(-3, 0, (n,), generator=g, device="cuda").float() for n in (M, N))
    bias = torch.randint(-8, 9, (N,), generator=g, device="cuda").to(od) if epi != "none" else torch.empty(0, dtype=od, device="cuda")
    v = (a.double() @ w.double().T).float()
    v = v * sa[:, None] * sb[None, :] if scaled else v
    v = v + bias.float() if epi != "none" else v
    want = (v.relu() if epi == "bias_relu" else v).to(od)
    c = torch.full((M + 2, N), -4096.0, dtype=od, device="cuda")
    raw = lambda t: t.to(td).view(torch.int8) if kind == "fp8" else t.to(td)
    f = compile_preshuffle_gemm(N=N, K=K, tile_m=64, tile_n=128, tile_k=64 if scaled else 32, in_dtype=kind, out_dtype=out, epilogue=epi)
    f.launch_forced(c[:M], raw(a), layout.shuffle_weight(raw(w)).contiguous(), sa if scaled else None, sb if scaled else None, bias, M, N, None, force_path=1, tile=(64, 64), splits=splits)
    torch.cuda.synchronize()
    assert torch.equal(c[:M], want)
    assert (c[M:] == -4096.0).all()
