"""The tile order the tiled kernel walks (psg_tile_order, evaluated on the device for every workgroup id) against
the oracle's restatement of the reference's xcd_remap_bx_by (kernels/common/mma/mfma_preshuffle_pipeline.py:685-729),
bit-exact, including ragged grids."""

import numpy as np
import pytest
import torch

from oracle import psg_oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("tiles_m,tiles_n,group_m", [(32, 16, 8), (64, 112, 8), (7, 5, 3), (3, 4, 2), (1, 13, 8), (13, 1, 4),
                                                      (17, 9, 16), (5, 5, 1), (41, 28, 8)])
def test_device_tile_order_equals_oracle(tiles_m, tiles_n, group_m):
    from flydsl_amd import _lib

    handle = _lib.lib()
    out = torch.full((tiles_m * tiles_n, 2), -1, dtype=torch.int32, device="cuda")
    rc = handle.psg_debug_tile_order(tiles_m, tiles_n, group_m, out.data_ptr(), _lib.stream_handle(None))
    assert rc == 0, handle.psg_last_error()
    torch.cuda.synchronize()
    got = out.cpu().numpy()
    want = np.array([O.xcd_remap_bx_by(i // tiles_n, i % tiles_n, tiles_m * 128, tile_m=128, tile_n=256, n=tiles_n * 256,
                                       xcd_swizzle=group_m) for i in range(tiles_m * tiles_n)], dtype=np.int32)
    assert np.array_equal(got, want)
    assert len({(int(a), int(b)) for a, b in got}) == tiles_m * tiles_n


@pytest.mark.parametrize("kind,M,N,K", [("int8", 4096, 8192, 128), ("fp8", 4001, 8192, 128), ("bf16", 4096, 4112, 64), ("fp4", 4096, 8192, 256), ("fp4", 8161, 4096, 512)])
def test_the_librarys_order_changes_no_bit(kind, M, N, K):
    """More tiles than CUs, aligned so that groups of 8 start every XCD at the same columns: the default order is another one."""
    from flydsl_amd import layout
    from flydsl_amd.kernels.gemm.mxfp4_preshuffle import launch_gemm
    from flydsl_amd.kernels.gemm.preshuffle_gemm import compile_preshuffle_gemm

    g = torch.Generator(device="cuda").manual_seed(K)
    st = torch.cuda.current_stream()
    out = [torch.full((M + 3, N), 9.0, dtype=torch.bfloat16, device="cuda") for _ in range(2)]
    u8 = lambda *shape: torch.randint(0, 256, shape, generator=g, device="cuda", dtype=torch.uint8)
    if kind == "fp4":
        a, b = u8(M, K // 2), u8(N, K // 2)
        sa, sb = (torch.randint(120, 130, ((r + 31) // 32 * 32, K // 32), generator=g, device="cuda", dtype=torch.uint8) for r in (M, N))
        for c, swizzle in zip(out, (0, 8)):
            launch_gemm(c, a, b, sa, sb, M, N, st, N, K, 64, 256, 256, "fp4", "bf16", "fp4", 1, -1, -1, -1, -1, -1, -1, 2, swizzle)
    else:
        td = {"int8": torch.int8, "fp8": torch.float8_e4m3fn, "bf16": torch.bfloat16}[kind]
        x = [torch.randn(r, K, generator=g, device="cuda").mul_(20) for r in (M, N)]
        a, b = (v.round().to(td) if kind == "int8" else v.to(td) for v in x)
        sa, sb = (torch.rand(r, generator=g, device="cuda") for r in (M, N))
        for c, swizzle in zip(out, (0, 8)):
            f = compile_preshuffle_gemm(N=N, K=K, tile_m=128, tile_n=256, tile_k=64, in_dtype=kind, xcd_swizzle=swizzle)
            f(c[:M].view(-1), a, b, sa, sb, torch.empty(0, dtype=torch.bfloat16, device="cuda"), M, N, st)
    torch.cuda.synchronize()
    assert torch.equal(out[0].view(torch.int16), out[1].view(torch.int16)) and (out[0][M:] == 9.0).all() and not (out[0][:M] == 9.0).all(1).any()
