"""Either side of the lines at which a problem of few rows leaves the kernel that streams W for the tiles: the columns that make one round of the
CUs (33 to 64 rows), rows of 4 to 8 KB (65 to 256 rows); and sizes whose large tile the estimated time decides.  The automatic plan against the general tiled path of the same problem.

int8 sums are whole numbers, so those results are the same bits; of the other kinds the two fp32 sums differ by their order alone, and a result by one
rounding to 16 bits at most."""

import pytest
import torch

from flydsl_amd import _lib
from flydsl_amd.kernels.gemm.preshuffle_gemm import compile_preshuffle_gemm
from flydsl_amd.kernels.gemm.mxfp4_preshuffle import launch_gemm

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", ["int8", "fp8", "bf16", "fp16"])
@pytest.mark.parametrize("M,N,KB", [
    (33, 8192, 512), (33, 8208, 512), (64, 8224, 64), (64, 8224, 1088), (40, 9216, 6144), (33, 16400, 2048), (64, 66048, 128),
    (65, 1024, 4224), (129, 1040, 8128), (256, 1024, 4160), (65, 1008, 4224), (192, 1360, 4992),
    # (the large tiles, by their estimated times)
    (4329, 1840, 1856), (1614, 4896, 1664), (411, 16720, 2944), (3683, 2288, 1088), (617, 11008, 1536),
])
def test_lines(dtype, M, N, KB):
    K = KB // 2 if dtype in ("bf16", "fp16") else KB
    g = torch.Generator(device="cuda")
    g.manual_seed(M + N)
    if dtype in ("bf16", "fp16"):
        td = torch.bfloat16 if dtype == "bf16" else torch.float16
        a, b = (torch.randn(r, K, generator=g, device="cuda").to(td) for r in (M, N))
        sa = sb = None
    else:
        a, b = (torch.randint(-60, 61, (r, K), generator=g, device="cuda", dtype=torch.int8) for r in (M, N))  # finite as fp8 too
        if dtype == "fp8":
            a, b = a.view(torch.float8_e4m3fn), b.view(torch.float8_e4m3fn)
        sa, sb = (torch.rand(r, generator=g, device="cuda") * 0.01 + 0.001 for r in (M, N))
    out = "fp16" if dtype == "fp16" else "bf16"
    to = torch.float16 if dtype == "fp16" else torch.bfloat16
    bias = torch.randn(N, generator=g, device="cuda").to(to)
    fn = compile_preshuffle_gemm(N=N, K=K, tile_m=64, tile_n=256, tile_k=64 * K // KB, in_dtype=dtype, out_dtype=out, epilogue="bias_relu")
    got, want = (torch.full((M + 16, N), -8192.0, dtype=to, device="cuda") for _ in range(2))
    fn(got, a, b, sa, sb, bias, M, N, torch.cuda.current_stream())
    fn.launch_forced(want, a, b, sa, sb, bias, M, N, torch.cuda.current_stream(), force_path=1, tile=(32, 256))
    torch.cuda.synchronize()
    assert (got[M:] == -8192.0).all()
    if dtype == "int8":
        assert torch.equal(got[:M], want[:M])
    else:
        x, y = got[:M].float(), want[:M].float()
        assert ((x - y).abs() <= 2.0 ** (-10 if dtype == "fp16" else -7) * y.abs() + 1e-5 * y.abs().max()).all()
    # what the tiles took over from the streaming kernel goes without a workspace, as it did there
    if M <= 64:
        assert _lib.lib().psg_workspace_bytes(M, N, K, _lib.IN_DTYPE[dtype]) == 0


@pytest.mark.parametrize("M,N,K", [(33, 8192, 2048), (33, 8224, 2048), (48, 10240, 8192), (64, 8224, 2304), (36, 24576, 2048)])
def test_fp4_lines(M, N, K):
    g = torch.Generator(device="cuda")
    g.manual_seed(M + N)

    def data(lo, hi, *shape):
        return torch.randint(lo, hi, shape, generator=g, device="cuda", dtype=torch.uint8)

    a, b = data(0, 256, M, K // 2), data(0, 256, N, K // 2)
    sa, sb = data(120, 130, (M + 31) // 32 * K), data(120, 130, N // 32 * K)
    got, want = (torch.full((M + 16, N), -8192.0, dtype=torch.bfloat16, device="cuda") for _ in range(2))
    for c, path in ((got, 0), (want, 3)):
        launch_gemm(c, a, b, sa, sb, M, N, torch.cuda.current_stream(), N, K, 64, 128, 256, "fp4", "bf16", "fp4", 1, -1, -1, -1, -1, -1, -1, 0, 0, _force_path=path)
    torch.cuda.synchronize()
    assert (got[M:] == -8192.0).all()
    x, y = got[:M].float(), want[:M].float()
    assert ((x - y).abs() <= 2.0 ** -7 * y.abs() + 1e-5 * y.abs().max()).all()
    assert _lib.lib().psg_workspace_bytes(M, N, K, 4) == 0
