"""Operands and outputs of more than 4 GiB, which a descriptor of 32 bits no longer holds.  C: the large tiles store it through descriptors and redirect what lies past N out of their
bounds; the small tiles store by 64-bit addresses and have the same sums, so every bit has to be the same.  A: half steps past a row."""

import ctypes

import pytest
import torch

pytestmark = pytest.mark.gpu

KINDS = {"int8": torch.int8, "fp8": torch.float8_e4m3fn, "fp16": torch.float16, "bf16": torch.bfloat16, "fp4": None}


def _compare(kind, tile, M, N, K):
    from flydsl_amd import _lib

    g = torch.Generator(device="cuda").manual_seed(N)
    mx, td = kind == "fp4", KINDS[kind]
    if mx:
        a, b = (torch.randint(0, 256, (r, K // 2), generator=g, device="cuda", dtype=torch.uint8) for r in (M, N))
        sa, sb = (torch.randint(120, 130, ((r + 31) // 32 * 32 * (K // 32),), generator=g, device="cuda", dtype=torch.uint8) for r in (M, N))
    else:
        a, b = (torch.randint(-8, 9, (r, K), generator=g, device="cuda", dtype=torch.int8).to(td) for r in (M, N))
        sa, sb = (torch.rand(r, generator=g, device="cuda") for r in (M, N))
    handle = _lib.lib()

    def run(tile_m, tile_n):
        c = torch.full((M, N), -7.0, dtype=torch.bfloat16, device="cuda")
        args = _lib.MxArgs() if mx else _lib.A8W8Args()
        args.c, args.a, args.b = c.data_ptr(), a.data_ptr(), b.data_ptr()
        if kind in ("int8", "fp8", "fp4"):
            args.scale_a, args.scale_b = sa.data_ptr(), sb.data_ptr()
        args.M, args.N, args.K = M, N, K
        if not mx:
            args.in_dtype = list(KINDS).index(kind)
        args.force_path, args.tile_m, args.tile_n, args.tile_k, args.reserved = 1, tile_m, tile_n, 1, 8 if (tile_m, tile_n) == (256, 256) else 0
        rc = (handle.psg_gemm_mxfp4 if mx else handle.psg_gemm_a8w8)(ctypes.byref(args), _lib.stream_handle(None))
        assert rc == 0, handle.psg_last_error()
        torch.cuda.synchronize()
        return c

    want = run(64, 256 if mx else 64)
    for _ in range(2):
        assert torch.equal(run(*tile).view(torch.int64), want.view(torch.int64))


# 4.98 GB, half a tile of columns past N: from row tile 0 on, 4 GiB ahead lie rows of C that another XCD works on at the same time
@pytest.mark.parametrize("kind,tile", [(k, t) for k in KINDS for t in ((128, 256), (256, 256)) if (k, t) != ("fp4", (256, 256))])
def test_columns_past_n_are_dropped(kind, tile):
    _compare(kind, tile, 16384, 151936, 256 if kind == "fp4" else 64)


@pytest.mark.parametrize("tile", [(64, 64), (128, 128), (128, 256), (256, 256)])
def test_half_steps_past_a_row_of_more_than_4_gib_of_a_read_zero(tile):
    """A row of an odd number of half steps: the missing half is fetched from past the bounds, where an infinity of another row must not be found."""
    from flydsl_amd import _lib

    M, N, K = 65536, 256, 32800
    a = torch.full((M, K), 0.25, dtype=torch.bfloat16, device="cuda")
    at = 0xFFFFFFF0 // 2
    a.view(-1)[at:at + 8] = float("inf")
    b = torch.ones(N, K, dtype=torch.bfloat16, device="cuda")
    c = torch.zeros(M, N, dtype=torch.bfloat16, device="cuda")
    args = _lib.A8W8Args()
    args.c, args.a, args.b, args.M, args.N, args.K, args.in_dtype = c.data_ptr(), a.data_ptr(), b.data_ptr(), M, N, K, 3
    args.force_path, args.tile_m, args.tile_n, args.tile_k, args.reserved = 1, *tile, 1, 8 if tile == (256, 256) else 0
    handle = _lib.lib()
    assert handle.psg_gemm_a8w8(ctypes.byref(args), _lib.stream_handle(None)) == 0, handle.psg_last_error()
    torch.cuda.synchronize()
    want = torch.full((M,), K * 0.25, device="cuda").bfloat16()
    want[at // K] = float("inf")
    assert torch.equal(c, want[:, None].expand(M, N))


# 2^25 columns: 64 MiB a row of C, so that a tile of 128 rows spans 8 GiB
@pytest.mark.parametrize("kind,tile,M,N,K", [("int8", (128, 256), 128, 1 << 25, 64), ("bf16", (128, 256), 100, 1 << 25, 32), ("int8", (256, 256), 200, (1 << 24) + 16, 64),
                                             ("fp4", (128, 256), 128, (1 << 25) - 32, 256)])
def test_rows_further_apart_than_32_bits(kind, tile, M, N, K):
    _compare(kind, tile, M, N, K)
