"""Workspace of an MX product, by its sizes (no GPU): asked for where the general kernel's K splits are what runs, and nowhere else."""

import pytest

from flydsl_amd.kernels.gemm.mxfp4_preshuffle import _plan


def _need(M, N, K, fa, fb, path=0, batch=1):
    return _plan(M, N, N, K, 64, 128, 256, fa, "bf16", fb, batch, -1, -1, -1, -1, -1, -1, 0, path, None, 0, 1, False)[2]


@pytest.mark.parametrize("M,N,K,fa,fb,splits", [
    (16, 4096, 4096, "fp8", "fp4", 0), (16, 512, 8192, "fp8", "fp8", 8), (33, 992, 14336, "fp8", "fp8", 4),  # fewer columns than the small-M kernel is for
    (33, 9248, 4352, "fp8", "fp4", 0), (38, 14112, 5376, "fp6", "fp4", 0), (56, 9504, 7936, "fp8", "fp4", 0),  # small-M, two rounds
    (33, 8224, 4352, "fp8", "fp8", 2), (44, 15232, 8448, "fp8", "fp8", 2), (38, 10112, 9984, "fp8", "fp4", 4), (65, 7168, 8704, "fp6", "fp4", 2), (47, 11456, 8448, "fp8", "fp4", 2),
    (67, 9568, 8960, "fp8", "fp8", 0), (97, 11008, 13824, "fp8", "fp4", 0), (82, 13920, 13056, "fp8", "fp8", 0), (94, 6400, 7424, "fp8", "fp4", 0),  # more splits than pay: tiles, small-M
    (64, 8192, 8192, "fp4", "fp8", 0), (64, 8192, 8192, "fp6", "fp8", 0), (64, 512, 8192, "fp4", "fp8", 2)])
def test_workspace_is_asked_for_where_it_is_used(M, N, K, fa, fb, splits):
    assert _need(M, N, K, fa, fb) == splits * M * N * 4
    assert _need(M, N, K, fa, fb, batch=2) == 0


def test_the_general_kernel_alone_wants_its_splits_anywhere():
    assert _need(33, 9248, 4352, "fp8", "fp4", path=3) == 2 * 33 * 9248 * 4
    assert _need(97, 11008, 13824, "fp8", "fp4", path=3) == 2 * 97 * 11008 * 4
