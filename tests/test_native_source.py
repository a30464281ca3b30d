"""What csrc/native.cpp does while the interpreter's lock is given up, by its text (the mistake it guards against ends the process, so it
is not made to happen): nothing but the call into the library, and the lock is taken back on every way out."""

import os
import re

import pytest

import flydsl_amd

SOURCE = os.path.join(os.path.dirname(flydsl_amd.__file__), "csrc", "native.cpp")


def _without_comments():
    return re.sub(r"//[^\n]*", "", open(SOURCE).read())


def _bodies(text):
    """The argument of every released(...) call."""
    for m in re.finditer(r"return released\(", text):
        depth, i = 1, m.end()
        while depth:
            depth += {"(": 1, ")": -1}.get(text[i], 0)
            i += 1
        yield text[m.end():i - 1]


def test_no_tensor_is_touched_without_the_lock():
    bodies = list(_bodies(_without_comments()))
    assert len(bodies) == 5
    for body in bodies:
        # a tensor's members may throw, materialise a copy-on-write storage or change under another thread
        assert "->" not in body and "data_ptr" not in body and "x_code" not in body and "Py" not in body, body


def test_the_lock_comes_back_when_something_throws():
    # the macros restore the thread state only where the block is left at its end
    assert "Py_BEGIN_ALLOW_THREADS" not in _without_comments()


def test_without_the_extension_the_python_checks_do_it():
    """The extension spares a launch its host time and nothing else: where it does not load, a warning names the cause and the calls go on."""
    import subprocess
    import sys

    code = """
import sys, warnings
sys.modules["flydsl_amd._native"] = None  # what an extension that is not built, or built against another torch, looks like
import pytest, torch
from flydsl_amd import _lib, quant_device
from flydsl_amd.kernels.gemm.mxfp4_preshuffle import launch_gemm
from flydsl_amd.kernels.moe.moe_gemm_2stage import compile_moe_reduction
from flydsl_amd.kernels.moe.mxfp_moe import moe_mxfp4_sort
z = lambda *s, dt=torch.uint8: torch.zeros(*s, dtype=dt)
x = z(32, 256, dt=torch.bfloat16)
with pytest.raises(ValueError, match="device tensor"), pytest.warns(RuntimeWarning, match="_native.so"):
    quant_device.pertoken_quant(x, torch.int8, stream=7, out=(z(32, 256), z(32, dt=torch.float32)))
warnings.simplefilter("error")  # once is enough
with pytest.raises(ValueError, match="device tensor"):
    quant_device.per_1x32_f4_quant(x, stream=7, out=(z(32, 128), z(32, 8)))
with pytest.raises(ValueError, match="device tensor"):
    launch_gemm(z(32, 64), z(32, 128), z(64, 128), z(32, 8), z(64, 8), 32, 64, 7, 64, 256, 64, 128, 256, "fp4", "bf16", "fp4", 1, -1, -1, -1, -1, -1, -1, 0, 0)
with pytest.raises(ValueError, match="device"):
    compile_moe_reduction(topk=2, model_dim=64, dtype_str="bf16")(x, x, None, None, 64, 7)
with pytest.raises(TypeError, match="device tensor"):
    moe_mxfp4_sort(z(32, 8), z(32), z(2), 32, out=z(32, 8), stream=7)
"""
    done = subprocess.run([sys.executable, "-c", code], cwd=os.path.dirname(os.path.dirname(flydsl_amd.__file__)), capture_output=True, text=True)
    assert done.returncode == 0, done.stderr


def test_operands_that_are_no_tensors_get_the_errors_of_the_checks():
    import pytest
    import torch

    from flydsl_amd.kernels.moe.moe_gemm_2stage import compile_moe_gemm1
    from flydsl_amd.kernels.moe.moe_sorting import moe_softmax_sort_flydsl
    from flydsl_amd.kernels.moe.mxfp_moe import flydsl_mxfp4_gemm1, flydsl_mxfp4_gemm2
    from flydsl_amd.quant_device import per_1x32_f4_quant, pertoken_quant

    t = torch.zeros(64, dtype=torch.int32)
    stage = compile_moe_gemm1(model_dim=256, inter_dim=128, experts=2, topk=1, tile_m=16, tile_n=64, tile_k=128, doweight_stage1=False, in_dtype="int8")
    for ids in (None, [0, 1], 4096):
        with pytest.raises(ValueError, match="device"):
            stage(t, t, t, t, t, ids, t, t, t, 3, 128, 256, 2, 7)
        with pytest.raises(ValueError, match="device tensor"):
            moe_softmax_sort_flydsl(torch.zeros(4, 8), ids, t, t, t, None, 8, 2, "f32", stream=7)
        kw = dict(cumsum_tensor=t, BM=32, NE=2, D_HIDDEN=256, D_INTER=256, topk=1, stream=7)
        u8 = t.view(torch.uint8)
        with pytest.raises(TypeError, match="m_indices"):
            flydsl_mxfp4_gemm1(a_quant=u8, a_scale_sorted_shuffled=u8, w1_u8=u8, w1_scale_u8=u8, sorted_expert_ids=t, m_indices=ids, inter_sorted_quant=u8,
                               inter_sorted_shuffled_scale=u8, n_tokens=3, **kw)
        with pytest.raises(TypeError, match="device tensor"):
            flydsl_mxfp4_gemm2(inter_sorted_quant=u8, inter_sorted_shuffled_scale=u8, w2_u8=u8, w2_scale_u8=u8, sorted_expert_ids=ids, sorted_token_ids=t, sorted_weights=t,
                               flat_out=t.bfloat16(), M_logical=3, max_sorted=64, epilog="atomic", **kw)
        with pytest.raises(ValueError, match="device tensor"):  # the clear buffer, the workspace; numbers that are no plain ones
            moe_softmax_sort_flydsl(torch.zeros(4, 8), t, t, t, t, ids, 8, 2, "f32", workspace=False if ids is None else ids, stream=7)
    with pytest.raises(ValueError, match="device tensor"):
        moe_softmax_sort_flydsl(torch.zeros(4, 8), t, t, t, t, None, 8, 2, "f32", renormalize=t, stream=7)
    with pytest.raises(ValueError, match="one element"):
        stage(t, t, t, t, t, t, t, t, t, 3, t, 256, 2, 7)
    x = torch.zeros(4, 64)
    for out in (7, "y", t, {}):
        with pytest.raises(ValueError, match="device tensor"):
            pertoken_quant(x, torch.int8, stream=7, out=out)
        with pytest.raises(ValueError, match="device tensor"):
            per_1x32_f4_quant(x, stream=7, out=out)
    with pytest.raises(ValueError, match="device tensor"):
        pertoken_quant(x, [torch.int8], stream=7, out=(t, t))
    with pytest.raises(ValueError, match="device tensor"):
        per_1x32_f4_quant(x, shuffle=t, stream=7, out=(t, t))
    with pytest.raises(NotImplementedError):
        flydsl_mxfp4_gemm2(inter_sorted_quant=u8, inter_sorted_shuffled_scale=u8, w2_u8=u8, w2_scale_u8=u8, sorted_expert_ids=t, sorted_token_ids=t, sorted_weights=t,
                           flat_out=t.bfloat16(), M_logical=3, max_sorted=64, epilog=["atomic"], **kw)


def test_scratch_is_not_asked_for_before_the_output_is_looked_at():
    import numpy as np
    import pytest
    import torch

    from flydsl_amd.kernels.gemm.mxfp4_preshuffle import launch_gemm

    u8 = torch.zeros(64, dtype=torch.uint8)
    for c, error in ((u8, ValueError), (np.zeros(64), TypeError)):  # 33 x 992 x 14336 splits K and needs scratch
        with pytest.raises(error):
            launch_gemm(c, u8, u8, u8, u8, 33, 992, 7, 992, 14336, 64, 128, 256, "fp8", "bf16", "fp4", 1, -1, -1, -1, -1, -1, -1, 0, 0)


@pytest.mark.parametrize("big", [2**40, 2**60, 2**70, -2**62, -2**70])
def test_numbers_beyond_any_size_get_the_errors_of_the_checks(big):
    import torch

    from flydsl_amd.kernels.gemm.mxfp4_preshuffle import launch_gemm
    from flydsl_amd.kernels.moe.moe_gemm_2stage import compile_moe_gemm1
    from flydsl_amd.kernels.moe.mxfp_moe import flydsl_mxfp4_gemm1, flydsl_mxfp4_gemm2

    t = torch.zeros(64, dtype=torch.int32)
    u8 = t.view(torch.uint8)
    stage = compile_moe_gemm1(model_dim=256, inter_dim=128, experts=2, topk=1, tile_m=16, tile_n=64, tile_k=128, doweight_stage1=False, in_dtype="int8")
    for tokens, blocks in ((big, 2), (3, big)):
        with pytest.raises(ValueError, match="device"):
            stage(t, t, t, t, t, t, t, t, t, tokens, 128, 256, blocks, 7)
    kw = dict(cumsum_tensor=t, BM=32, NE=2, D_HIDDEN=256, D_INTER=256, topk=1, stream=7)
    with pytest.raises(TypeError, match="device tensor"):
        flydsl_mxfp4_gemm1(a_quant=u8, a_scale_sorted_shuffled=u8, w1_u8=u8, w1_scale_u8=u8, sorted_expert_ids=t, m_indices=t, inter_sorted_quant=u8,
                           inter_sorted_shuffled_scale=u8, n_tokens=big, **kw)
    with pytest.raises(TypeError, match="device tensor"):
        flydsl_mxfp4_gemm2(inter_sorted_quant=u8, inter_sorted_shuffled_scale=u8, w2_u8=u8, w2_scale_u8=u8, sorted_expert_ids=t, sorted_token_ids=t, sorted_weights=t.float(),
                           flat_out=t.bfloat16(), M_logical=big, max_sorted=64, epilog="atomic", **kw)
    with pytest.raises(ValueError, match="device tensor"):
        launch_gemm(u8, u8, u8, u8, u8, big, 64, 7, 64, 256, 64, 128, 256, "fp4", "bf16", "fp4", 1, -1, -1, -1, -1, -1, -1, 0, 0)
