"""The 128x256 tile of the 8- and 16-bit GEMM at the edges of its loop and of its tile: rows around 128, columns that end in the first, second and last
wavefront, rows of W of one half step up and with and without a half step at the end, K splits, W row-major.

Operands are multiples of 1/4 up to 2 (int8: integers up to 8) and scales powers of two, so every sum is exact in fp32 and the result has one right value."""

import ctypes

import pytest
import torch

pytestmark = pytest.mark.gpu

KINDS = {"int8": torch.int8, "fp8": torch.float8_e4m3fn, "fp16": torch.float16, "bf16": torch.bfloat16}


@pytest.mark.parametrize("rowmajor", [False, True], ids=["preshuffled", "rowmajor"])
@pytest.mark.parametrize("kind", list(KINDS))
@pytest.mark.parametrize("M,N,kbytes,splits", [(1, 16, 64, 1), (127, 256, 128, 1), (128, 272, 192, 1), (129, 240, 256, 1), (255, 528, 320, 1), (257, 80, 576, 1),
                                               (384, 1040, 1088, 1), (130, 336, 1088, 2), (200, 272, 1984, 3), (1100, 784, 2112, 1)])
def test_edges(M, N, kbytes, splits, kind, rowmajor):
    from flydsl_amd import _lib, layout

    dev, td, wide = torch.device("cuda"), KINDS[kind], kind in ("fp16", "bf16")
    K = kbytes // 2 if wide else kbytes
    g = torch.Generator(device="cuda").manual_seed(M + kbytes)
    a, w = (torch.randint(-8, 9, (r, K), generator=g, device="cuda").float() * (1.0 if kind == "int8" else 0.25) for r in (M, N))
    sa, sb = (2.0 ** torch.randint(-5, -2, (n,), generator=g, device="cuda").float() for n in (M, N))
    aq, wq = a.to(td), w.to(td)
    b = wq.contiguous() if rowmajor else layout.shuffle_weight(wq.view(torch.int8) if kind == "fp8" else wq).contiguous()
    v = (a.double() @ w.double().T).float()
    want = (v if wide else v * sa[:, None] * sb[None, :]).to(torch.bfloat16)
    c = torch.full((M + 3, N), -8192.0, dtype=torch.bfloat16, device=dev)
    ws = torch.empty(splits * M * N * 4, dtype=torch.uint8, device=dev)
    args = _lib.A8W8Args()
    args.c, args.a, args.b = c.data_ptr(), aq.data_ptr(), b.data_ptr()
    if not wide:
        args.scale_a, args.scale_b = sa.data_ptr(), sb.data_ptr()
    args.M, args.N, args.K, args.in_dtype, args.b_layout = M, N, K, list(KINDS).index(kind), int(rowmajor)
    args.force_path, args.tile_m, args.tile_n, args.tile_k = 1, 128, 256, splits
    args.workspace, args.workspace_bytes = ws.data_ptr(), ws.numel()
    handle = _lib.lib()
    rc = handle.psg_gemm_a8w8(ctypes.byref(args), _lib.stream_handle(None))
    assert rc == 0, handle.psg_last_error()
    torch.cuda.synchronize()
    assert torch.equal(c[:M], want)
    assert (c[M:] == -8192.0).all()
