"""The planner's own choice between the two large tiles, on both sides of the line that keeps 256x256 tiles making one round of the CUs: as many rows as share W, 128x256 tiles one and
a half to a CU, 256x256 tiles half a round and more than one.

Operands are whole numbers and scales powers of two, so every sum is exact in fp32 and the result has one right value."""

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind,M,N,K", [("int8", 1536, 9248, 320), ("int8", 1537, 8976, 320), ("bf16", 2048, 5632, 160), ("bf16", 2049, 5904, 160), ("fp16", 1100, 11056, 96),
                                        ("int8", 1800, 4624, 448), ("int8", 1801, 4352, 448), ("bf16", 4097, 4112, 96)])
def test_large_tiles(kind, M, N, K):
    from flydsl_amd import layout
    from flydsl_amd.kernels.gemm.preshuffle_gemm import compile_preshuffle_gemm

    td = {"int8": torch.int8, "fp16": torch.float16, "bf16": torch.bfloat16}[kind]
    g = torch.Generator(device="cuda").manual_seed(M + N)
    a, w = (torch.randint(-4, 5, (r, K), generator=g, device="cuda") for r in (M, N))
    sa, sb = (2.0 ** torch.randint(-5, -2, (n,), generator=g, device="cuda").float() for n in (M, N))
    v = (a.double() @ w.double().T).float()
    want = (v * sa[:, None] * sb[None, :] if kind == "int8" else v).bfloat16()
    c = torch.full((M + 3, N), -8192.0, dtype=torch.bfloat16, device="cuda")
    f = compile_preshuffle_gemm(N=N, K=K, tile_m=64, tile_n=128, tile_k=64 if kind == "int8" else 32, in_dtype=kind)
    f(c[:M].view(-1), a.to(td), layout.shuffle_weight(w.to(td)).contiguous(), sa, sb, torch.empty(0, dtype=torch.bfloat16, device="cuda"), M, N, torch.cuda.current_stream())
    torch.cuda.synchronize()
    assert torch.equal(c[:M], want)
    assert (c[M:] == -8192.0).all()
