"""Problems on the lines of the tile choice for int8 and 16-bit operands, as the planner launches them: few rows of tiles, one round of 256x256 tiles, nine rows of 64x256 tiles, weights beyond the
last-level cache.

Operands are whole numbers and scales powers of two, so every sum is exact in fp32 and the result has one right value."""

import ctypes

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind,M,N,K,tile", [
    ("int8", 1025, 9024, 1600, (256, 256)), ("int8", 1026, 9024, 1152, (128, 256)), ("bf16", 769, 12304, 576, (256, 256)), ("bf16", 511, 17664, 1248, (256, 256)),
    ("int8", 838, 9248, 1088, (128, 128)), ("int8", 520, 13072, 1536, (64, 256)), ("fp16", 264, 11872, 544, (64, 256)), ("int8", 513, 28304, 6976, (128, 256)), ("bf16", 452, 16896, 8192, (256, 256))])
def test_planned_launch(kind, M, N, K, tile):
    from flydsl_amd import _lib, layout
    from flydsl_amd.kernels.gemm.preshuffle_gemm import compile_preshuffle_gemm

    out = [ctypes.c_int32() for _ in range(3)]
    assert _lib.lib().psg_debug_plan(M, N, K, {"int8": 0, "fp16": 2, "bf16": 3}[kind], *[ctypes.byref(v) for v in out]) == 0
    assert tuple(v.value for v in out) == (*tile, 1)
    td = {"int8": torch.int8, "fp16": torch.float16, "bf16": torch.bfloat16}[kind]
    g = torch.Generator(device="cuda").manual_seed(M + N)
    a, w = (torch.randint(-4, 5, (r, K), generator=g, device="cuda").to(td) for r in (M, N))
    sa, sb = (2.0 ** torch.randint(-5, -2, (n,), generator=g, device="cuda").float() for n in (M, N))
    v = torch.cat([a.double() @ part.double().T for part in w.split(4096)], 1).float()
    want = (v * sa[:, None] * sb[None, :] if kind == "int8" else v).bfloat16()
    c = torch.full((M + 3, N), -8192.0, dtype=torch.bfloat16, device="cuda")
    f = compile_preshuffle_gemm(N=N, K=K, tile_m=64, tile_n=128, tile_k=64 if kind == "int8" else 32, in_dtype=kind)
    f(c[:M].view(-1), a, layout.shuffle_weight(w).contiguous(), sa, sb, torch.empty(0, dtype=torch.bfloat16, device="cuda"), M, N, torch.cuda.current_stream())
    torch.cuda.synchronize()
    assert torch.equal(c[:M], want)
    assert (c[M:] == -8192.0).all()
