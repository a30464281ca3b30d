"""Fused epilogues and both output types on every tile of the tiled kernels, forced on ragged sizes (rows past M, columns past N).

Operands are multiples of 1/4 up to 2 and the scales powers of two, so the sums are exact in any order, and so is everything up to the bias;
silu and gelu add the error of an fp32 exponential and reciprocal, and every side rounds once to 16 bits."""

import pytest
import torch

pytestmark = pytest.mark.gpu

TILES = [((256, 256), 8), ((256, 256), 0), ((128, 256), 0), ((64, 256), 0), ((128, 128), 0), ((64, 64), 0)]
KINDS = {"fp8": torch.float8_e4m3fn, "int8": torch.int8, "bf16": torch.bfloat16, "fp16": torch.float16}


@pytest.mark.parametrize("out,half", [("bf16", 2.0 ** -8), ("fp16", 2.0 ** -11)])
@pytest.mark.parametrize("kind", list(KINDS))
@pytest.mark.parametrize("epilogue", ["none", "bias", "bias_relu", "bias_silu", "bias_gelu"])
def test_every_tile(kind, epilogue, out, half):
    from flydsl_amd import layout
    from kernels.gemm.preshuffle_gemm import compile_preshuffle_gemm

    M, N, K = 277, 272, 416
    wide = kind in ("bf16", "fp16")
    td, tout = KINDS[kind], torch.bfloat16 if out == "bf16" else torch.float16
    g = torch.Generator(device="cuda").manual_seed(len(epilogue))
    step = 1.0 if kind == "int8" else 0.25
    a, w = (torch.randint(-8, 9, (r, K), generator=g, device="cuda").float() * step for r in (M, N))
    if not wide:
        a, w = a[:, :384], w[:, :384]
    K = a.shape[1]
    scale = lambda n: 2.0 ** torch.randint(-5, -2, (n,), generator=g, device="cuda").float()
    sa, sb = (None, None) if wide else (scale(M), scale(N))
    bias = torch.randn(N, generator=g, device="cuda").to(tout)
    bias[:6] = torch.tensor([-0.0, 300.0, -300.0, 30000.0, -30000.0, -12.0], device="cuda").to(tout)  # both tails of the activations
    wq = w.to(td)
    shuffled = layout.shuffle_weight(wq.view(torch.int8) if kind == "fp8" else wq).view(td).contiguous()
    fn = compile_preshuffle_gemm(N=N, K=K, tile_m=64, tile_n=128, tile_k=32 if wide else 64, in_dtype=kind, out_dtype=out, epilogue=epilogue)
    v = a.double() @ w.double().T
    if not wide:
        v = v * sa.double()[:, None] * sb.double()[None, :]
    if epilogue != "none":
        v = (v.float() + bias.float()).double()  # the one rounding in front of the activation
    if epilogue == "bias_relu":
        v = v.clamp(min=0)
    if epilogue == "bias_silu":
        v = v / (1 + torch.exp(-v))
    if epilogue == "bias_gelu":
        v = 0.5 * v * (1 + torch.tanh(0.7978845608 * (v + 0.044715 * v ** 3)))
    for tile, layout_ in TILES:
        c = torch.full((M + 3, N), -8192.0, dtype=tout, device="cuda")
        fn.launch_forced(c, a.to(td).contiguous(), shuffled, sa, sb, bias, M, N, torch.cuda.current_stream(), force_path=1, tile=tile, wave_layout=layout_)
        assert (c[M:] == -8192.0).all(), tile
        if epilogue in ("bias_silu", "bias_gelu"):
            # half a unit in the last place of the output on top of the fp32 error (the exponent of exp2 is rounded to 24 bits: 2^-24 times
            # its size, at most 128); below the normal range of fp16 the spacing is 2^-24
            assert ((c[:M].double() - v).abs() <= (half + 2.0 ** -16) * v.abs() + 2.0 ** -24 + 1e-6).all(), tile
        else:
            assert torch.equal(c[:M], v.to(tout)), tile


@pytest.mark.parametrize("epilogue", ["bias_silu", "bias_gelu"])
def test_far_negative_tail(epilogue):
    """Divisors up to 2^128, whose reciprocals are below the normal range of fp32 while the product with v is not: silu(-88.5) = -3.3e-37."""
    from flydsl_amd import layout
    from kernels.gemm.preshuffle_gemm import compile_preshuffle_gemm

    M, N, K = 277, 272, 128
    bias = torch.zeros(N)
    bias[:40] = torch.arange(-88.5, -68.5, 0.5)
    bias[40:200] = torch.arange(-10.0, 0.0, 0.0625)
    bias[200:206] = torch.tensor([-1e30, 1e30, 1e38, -0.0, 1e-37, -1e-37])
    bias = bias.bfloat16().cuda()
    v = bias.double().expand(M, N)
    if epilogue == "bias_silu":
        want, exponent = torch.where(v < -88.7, 0.0, v * torch.sigmoid(v)), v.abs()
    else:
        y = 0.7978845608 * (v + 0.044715 * v ** 3)
        want, exponent = v * torch.sigmoid(2 * y), 2 * y.abs()
        want = torch.where(exponent > 88.7, torch.where(v > 0, v, 0.0), want)  # the divisor is past 2^128
    # half a unit of bf16, and 2^-23 times what goes into exp2 (two roundings), which is at most 128 where the result is not 0 or v
    rel = 2.0 ** -8 + 2.0 ** -22 * (1 + exponent.clamp(max=128))
    a, w = torch.zeros(M, K, device="cuda").to(torch.float8_e4m3fn), layout.shuffle_weight(torch.zeros(N, K, dtype=torch.int8, device="cuda")).view(torch.float8_e4m3fn)
    fn = compile_preshuffle_gemm(N=N, K=K, tile_m=64, tile_n=128, tile_k=64, in_dtype="fp8", out_dtype="bf16", epilogue=epilogue)
    for m, kw in [(M, dict(force_path=1, tile=tile, wave_layout=layout_)) for tile, layout_ in TILES] + [(16, dict(force_path=2)), (64, dict(force_path=2))]:
        c = torch.empty(m, N, dtype=torch.bfloat16, device="cuda")
        fn.launch_forced(c, a[:m], w, torch.ones(m, device="cuda"), torch.ones(N, device="cuda"), bias, m, N, torch.cuda.current_stream(), **kw)
        assert ((c.double() - want[:m]).abs() <= rel[:m] * want[:m].abs()).all(), kw
