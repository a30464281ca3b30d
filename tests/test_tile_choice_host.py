"""The planner's choice of a tile, by sizes (no GPU): what the estimates and the rules beside them say on both sides of their lines."""

import ctypes

import pytest

from flydsl_amd import _lib

KIND = {"int8": 0, "fp8": 1, "fp16": 2, "bf16": 3}


def _plan(kind, M, N, K):
    out = [ctypes.c_int32() for _ in range(3)]
    rc = _lib.lib().psg_debug_plan(M, N, K, KIND[kind], *[ctypes.byref(v) for v in out])
    assert rc == 0, _lib.lib().psg_last_error()
    return tuple(v.value for v in out)


@pytest.mark.parametrize("kind,M,N,K,tile", [
    ("int8", 838, 9248, 7296, (128, 128)), ("bf16", 806, 9280, 8192, (128, 128)), ("int8", 520, 13072, 1536, (64, 256)), ("bf16", 826, 9360, 1088, (64, 256)),
    ("int8", 1282, 6000, 6016, (64, 256)), ("fp16", 558, 13696, 1984, (64, 256))])
def test_smaller_tiles_of_the_smallest_estimate_stay(kind, M, N, K, tile):
    assert _plan(kind, M, N, K) == (*tile, 1)


@pytest.mark.parametrize("kind,M,N,K,rows", [
    ("int8", 1024, 9024, 4096, 256), ("int8", 1024, 8960, 4096, 128),  # 144 and 140 of 256 CUs
    ("int8", 1536, 6016, 4096, 256), ("int8", 1537, 5888, 4096, 128), ("int8", 1537, 6656, 4096, 256), ("bf16", 1536, 6016, 4096, 256), ("bf16", 1537, 6016, 4096, 128),  # rows that share W
    ("int8", 768, 12288, 2048, 256), ("int8", 1261, 8480, 1856, 256), ("int8", 941, 10048, 1856, 256), ("int8", 902, 10192, 1088, 128),
    ("int8", 1920, 6400, 6144, 256), ("int8", 2048, 6016, 6144, 128), ("int8", 2048, 6144, 4096, 128), ("bf16", 2048, 6144, 4096, 128),  # one and a half 128x256 tiles a CU: 375, 384
    ("int8", 1638, 5824, 704, 128), ("int8", 829, 10224, 832, 128), ("bf16", 2863, 4096, 192, 128), ("fp16", 717, 12320, 256, 128)])  # short rows
def test_large_tile_of_one_round(kind, M, N, K, rows):
    assert _plan(kind, M, N, K) == (rows, 256, 1)


@pytest.mark.parametrize("kind,M,N,K,rows", [("int8", 463, 17184, 4800, 256), ("int8", 463, 17104, 4800, 128), ("int8", 733, 11632, 4032, 256), ("int8", 733, 11456, 4032, 128), ("bf16", 511, 17664, 2496, 256),
                                             ("fp16", 720, 11696, 4352, 256), ("int8", 800, 8944, 6016, 128)])
def test_few_rows_of_tiles_on_little_more_than_half_of_the_cus(kind, M, N, K, rows):
    assert _plan(kind, M, N, K) == (rows, 256, 1)


@pytest.mark.parametrize("kind,M,N,K,rows", [
    ("int8", 3337, 21488, 13248, 256), ("int8", 2985, 23344, 13632, 256), ("int8", 3195, 20832, 14272, 256), ("bf16", 1113, 23744, 8320, 256), ("bf16", 1270, 22928, 7552, 256), ("fp16", 947, 28352, 8192, 256),
    ("int8", 4704, 18800, 12736, 128), ("int8", 4704, 18800, 12800, 256),  # 239.4 and 240.6 MB of W
    ("bf16", 2048, 20496, 5888, 256), ("bf16", 2049, 20496, 5888, 128),
    ("int8", 2624, 25376, 8384, 128), ("bf16", 1953, 27936, 4032, 128)])
def test_weights_beyond_the_last_level_cache(kind, M, N, K, rows):
    assert _plan(kind, M, N, K) == (rows, 256, 1)


@pytest.mark.parametrize("kind,M,N,K,tile", [("int8", 550, 14144, 12288, (64, 256)), ("int8", 550, 14144, 13312, (256, 256)), ("fp8", 540, 26688, 11648, (128, 256)),
                                             ("bf16", 556, 26928, 4480, (128, 256))])
def test_nine_rows_of_tiles_in_groups_of_eight(kind, M, N, K, tile):
    assert _plan(kind, M, N, K) == (*tile, 1)


@pytest.mark.parametrize("kind,M,N,K,tile", [
    ("fp16", 264, 11872, 1152, (64, 256)), ("bf16", 161, 20640, 1152, (64, 256)), ("bf16", 394, 8432, 1152, (64, 256)), ("bf16", 301, 11376, 1408, (64, 256)),  # at most one 128x256 tile a CU
    ("bf16", 703, 23456, 1792, (128, 256)), ("fp16", 909, 16400, 1536, (128, 256))])  # more
def test_16_bits_around_a_128x256_tile_a_cu(kind, M, N, K, tile):
    assert _plan(kind, M, N, K) == (*tile, 1)


def test_what_the_query_refuses():
    out = [ctypes.byref(ctypes.c_int32()) for _ in range(3)]
    h = _lib.lib()
    assert h.psg_debug_plan(16, 6144, 4096, 1, *out) == 0 and out[0]._obj.value == 0  # the streaming kernel
    for bad in ((0, 64, 64, 0), (64, 8, 64, 0), (64, 64, 0, 0), (64, 64, 64, 4), (64, 1 << 20, 1 << 20, 3)):
        assert h.psg_debug_plan(*bad, *out) != 0
    assert h.psg_debug_plan(64, 64, 64, 0, None, out[1], out[2]) != 0
