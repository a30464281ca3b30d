"""The planner's own choice on both sides of the lines that leave single tiles or builds out: one row of 64x64 tiles around a tile a CU (the builds that fetch W one and three steps
ahead), 16-bit problems around a 128x128 tile a CU, MXFP4 with 64x128 tiles one to a CU and 32x128 tiles more.

Operands are whole numbers and scales powers of two, so every sum is exact in fp32 and the result has one right value (MXFP4: the bits of the 64x256 tile, which adds up in the same order)."""

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind,M,N,K", [("int8", 33, 16384, 832), ("int8", 64, 16400, 832), ("int8", 35, 16448, 768), ("fp8", 48, 32768, 896), ("fp8", 64, 32832, 832), ("bf16", 34, 17216, 416),
                                        ("bf16", 1182, 3200, 480), ("bf16", 1408, 3328, 288), ("fp16", 2560, 1616, 544), ("bf16", 300, 10784, 352)])
def test_8_and_16_bits(kind, M, N, K):
    from flydsl_amd import layout
    from flydsl_amd.kernels.gemm.preshuffle_gemm import compile_preshuffle_gemm

    td = {"int8": torch.int8, "fp8": torch.float8_e4m3fn, "fp16": torch.float16, "bf16": torch.bfloat16}[kind]
    g = torch.Generator(device="cuda").manual_seed(M + N)
    a, w = (torch.randint(-4, 5, (r, K), generator=g, device="cuda") for r in (M, N))
    sa, sb = (2.0 ** torch.randint(-5, -2, (n,), generator=g, device="cuda").float() for n in (M, N))
    wq = layout.shuffle_weight(w.to(td).view(torch.int8) if kind == "fp8" else w.to(td)).contiguous()
    v = (a.double() @ w.double().T).float()
    want = (v * sa[:, None] * sb[None, :] if kind in ("int8", "fp8") else v).bfloat16()
    c = torch.full((M + 3, N), -8192.0, dtype=torch.bfloat16, device="cuda")
    f = compile_preshuffle_gemm(N=N, K=K, tile_m=64, tile_n=128, tile_k=32 if kind in ("fp16", "bf16") else 64, in_dtype=kind)
    f(c[:M].view(-1), a.to(td).view(torch.int8) if kind == "fp8" else a.to(td), wq, sa, sb, torch.empty(0, dtype=torch.bfloat16, device="cuda"), M, N, torch.cuda.current_stream())
    torch.cuda.synchronize()
    assert torch.equal(c[:M], want)
    assert (c[M:] == -8192.0).all()


@pytest.mark.parametrize("M,N,K", [(65, 10912, 768), (113, 10752, 1792), (129, 16416, 512), (315, 3264, 1024), (320, 5152, 1024), (33, 16512, 1024), (40, 20480, 1024), (64, 32800, 512)])
def test_mxfp4(M, N, K):
    from kernels.gemm.mxfp4_preshuffle import launch_gemm

    g = torch.Generator(device="cuda").manual_seed(M + N)
    u8 = lambda lo, hi, *shape: torch.randint(lo, hi, shape, generator=g, device="cuda", dtype=torch.uint8)
    a, b = u8(0, 256, M, K // 2), u8(0, 256, N, K // 2)
    sa, sb = u8(100, 150, (M + 31) // 32 * K), u8(100, 150, N // 32 * K)
    out = []
    for kw in (dict(_force_path=1, _tile=(64, 256)), {}):
        c = torch.full((M + 5, N), -7.0, dtype=torch.bfloat16, device="cuda")
        launch_gemm(c, a, b, sa, sb, M, N, None, N, K, 64, 128, 256, "fp4", "bf16", "fp4", 1, -1, -1, -1, -1, -1, -1, 0, 0, **kw)
        torch.cuda.synchronize()
        assert (c[M:] == -7.0).all()
        out.append(c[:M].view(torch.int16))
    assert torch.equal(*out)
