"""The kernel and tile that an fp4 x fp4, fp8 x fp8 or fp8 / fp6 x fp4 problem takes by itself: sizes on whose tile the estimate decides against the score, either side of
the lines between the small-M kernel, the general kernel's K splits and the tiles, ragged rows and columns, one tile and several rounds of them,
against the general MX kernel on the same operands.

Products of two codes and power-of-two scales are exact, so the two fp32 results differ by their order of summation alone: within 1e-5 of the largest.
The bf16 result is the fp32 one rounded once."""

import pytest
import torch

from flydsl_amd.kernels.gemm.mxfp4_preshuffle import launch_gemm

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("fmt,M,N,K,batch", [("fp4",) + s for s in [
    (48, 4096, 1024, 1), (64, 1024, 256, 1), (65, 1056, 1280, 1), (130, 2048, 1024, 1), (300, 7168, 2048, 1), (647, 6816, 1792, 1), (788, 5280, 4608, 1),
    (1163, 12384, 1280, 1), (4887, 4256, 1024, 1), (1285, 14048, 768, 1), (2127, 4384, 1536, 2),
]] + [("fp8",) + s for s in [
    (32, 8224, 512, 1), (33, 992, 512, 1), (33, 992, 14336, 1), (64, 8192, 1024, 1), (64, 8224, 1024, 1), (65, 32, 256, 1), (65, 4096, 512, 1), (128, 4128, 512, 1),
    (87, 8160, 4096, 1), (67, 9568, 8960, 1), (300, 992, 4096, 1), (383, 12384, 768, 1), (1164, 2880, 1024, 1), (4096, 1024, 512, 1), (2127, 4384, 1536, 2),
]] + [(f,) + s for f in ("fp8-fp4", "fp6-fp4") for s in [
    (32, 8224, 512, 1), (33, 992, 512, 1), (33, 992, 14336, 1), (64, 8192, 1024, 1), (64, 8224, 2304, 1), (64, 9248, 1024, 1), (65, 32, 256, 1), (128, 4128, 1536, 1),
    (300, 992, 4096, 1), (383, 12384, 768, 1), (1164, 2880, 1024, 1), (293, 14656, 1280, 1), (2311, 4544, 768, 1), (5000, 1024, 512, 1), (2127, 4384, 1536, 2),
]])
def test_planned_tile(fmt, M, N, K, batch):
    g = torch.Generator(device="cuda")
    g.manual_seed(M)
    chunks = (M + 31) // 32

    def data(lo, hi, *shape):
        return torch.randint(lo, hi, shape, generator=g, device="cuda", dtype=torch.uint8)

    fa, fb = (fmt, fmt) if "-" not in fmt else fmt.split("-")
    if fmt == "fp4":
        a, b = data(0, 256, batch, M, K // 2), data(0, 256, batch, N, K // 2)
    else:  # every finite positive and small negative code (0x7f and 0xff are NaN)
        a, b = data(0, 127, batch, M, K), data(0, 127, batch, N, K) if fb == "fp8" else data(0, 256, batch, N, K // 2)
        a[..., ::3] |= 128
    sa, sb = data(120, 130, batch, chunks * K), data(120, 130, batch, N // 32 * K)

    def run(path):
        c = torch.full((batch * M + 64, N), -8192.0, dtype=torch.bfloat16, device="cuda")
        launch_gemm(c, a, b, sa, sb, M, N, torch.cuda.current_stream(), N, K, 64, 128, 256, fa, "bf16", fb, batch, -1, -1, -1, -1, -1, -1, 0, 0,
                    _force_path=path)
        acc = torch.empty(batch, M, N, dtype=torch.float32, device="cuda")
        if batch == 1:
            launch_gemm(c, a, b, sa, sb, M, N, torch.cuda.current_stream(), N, K, 64, 128, 256, fa, "bf16", fb, 1, -1, -1, -1, -1, -1, -1, 0, 0,
                        _force_path=path, _acc=acc)
        torch.cuda.synchronize()
        assert (c[batch * M:] == -8192.0).all()
        return c[:batch * M].view(batch, M, N), acc

    (c, acc), (ref_c, ref) = run(0), run(3)
    if batch == 1 and fa == fb:  # (the others' tiles store no fp32)
        assert (acc - ref).abs().max() <= 1e-5 * ref.abs().max()
        if fmt == "fp4":
            assert torch.equal(c[0], acc[0].bfloat16())
    # the two fp32 sums may round to neighbouring bf16 values
    assert ((c.float() - ref_c.float()).abs() <= 2.0 ** -7 * ref_c.float().abs() + 1e-5 * ref_c.float().abs().max()).all()


@pytest.mark.parametrize("fmt,M,N,K", [("fp8",) + s for s in [  # 32x128, 64x128, 64x256, 128x256, 256x256 tiles
    (39, 32, 256), (101, 8416, 1024), (641, 9376, 512), (836, 8768, 1280), (1220, 9824, 1024)]] + [(f,) + s for f in ("fp8-fp4", "fp6-fp4") for s in [  # and 32x256
        (59, 32, 256), (393, 10048, 256), (644, 8864, 512), (802, 8736, 512), (554, 22080, 512), (1185, 10080, 256)]])
def test_planned_tile_in_fp16(fmt, M, N, K):
    """Builds of their own.  The scales keep the sums finite in fp16: 1280 products of up to 448 x 448 x 2^-18, 512 of 448 x 6 x 2^-7."""
    g = torch.Generator(device="cuda")
    g.manual_seed(N)

    def data(lo, hi, *shape):
        return torch.randint(lo, hi, shape, generator=g, device="cuda", dtype=torch.uint8)

    fa, fb = (fmt, fmt) if "-" not in fmt else fmt.split("-")
    a, b = data(0, 127, M, K), data(0, 127, N, K) if fb == "fp8" else data(0, 256, N, K // 2)
    a[..., ::3] |= 128
    sa, sb = data(112, 119, (M + 31) // 32 * K), data(112, 119, N // 32 * K) if fb == "fp8" else data(124, 130, N // 32 * K)
    out = []
    for path in (0, 3):
        c = torch.full((M + 64, N), -8192.0, dtype=torch.float16, device="cuda")
        launch_gemm(c, a, b, sa, sb, M, N, torch.cuda.current_stream(), N, K, 64, 128, 256, fa, "fp16", fb, 1, -1, -1, -1, -1, -1, -1, 0, 0, _force_path=path)
        assert (c[M:] == -8192.0).all()
        out.append(c[:M].float())
    c, ref = out
    assert ref.isfinite().all() and ref.abs().max() > 0.05
    # two fp32 sums of different order, each rounded to fp16 (subnormal from 2^-14 down)
    assert ((c - ref).abs() <= 2.0 ** -10 * ref.abs() + 2.0 ** -24 + 1e-5 * ref.abs().max()).all()


@pytest.mark.parametrize("fmt,M,N,K", [
    ("fp8-fp4", 33, 9248, 4352), ("fp6-fp4", 64, 8224, 8192), ("fp8-fp4", 38, 10112, 9984), ("fp6-fp4", 67, 9568, 8960), ("fp8-fp4", 94, 6400, 7424), ("fp6-fp4", 65, 8160, 1280),
    ("fp8-fp4", 33, 16416, 1792), ("fp8", 33, 8224, 4352), ("fp8", 51, 9440, 7680), ("fp8", 35, 9216, 1792), ("fp8", 65, 4096, 8448), ("fp8", 70, 8032, 9216)])
def test_with_and_without_a_workspace(fmt, M, N, K):
    """Either side of the lines between one and two rounds of the small-M kernel, the K splits and the tiles, ragged in rows and columns."""
    g = torch.Generator(device="cuda")
    g.manual_seed(M + N)
    fa, fb = (fmt, fmt) if "-" not in fmt else fmt.split("-")

    def data(lo, hi, *shape):
        return torch.randint(lo, hi, shape, generator=g, device="cuda", dtype=torch.uint8)

    a, b = data(0, 127, M, K), data(0, 127, N, K) if fb == "fp8" else data(0, 256, N, K // 2)
    a[..., ::3] |= 128
    sa, sb = data(120, 130, (M + 31) // 32 * K), data(120, 130, N // 32 * K)
    out = []
    for kw in (dict(), dict(_no_split=True), dict(_force_path=3, _no_split=True)):
        c = torch.full((M + 64, N), -8192.0, dtype=torch.bfloat16, device="cuda")
        launch_gemm(c, a, b, sa, sb, M, N, torch.cuda.current_stream(), N, K, 64, 128, 256, fa, "bf16", fb, 1, -1, -1, -1, -1, -1, -1, 0, 0, **kw)
        assert (c[M:] == -8192.0).all()
        out.append(c[:M].float())
    for c in out[:2]:  # fp32 sums of different order, which may round to neighbouring bf16 values
        assert ((c - out[2]).abs() <= 2.0 ** -7 * out[2].abs() + 1e-5 * out[2].abs().max()).all()
