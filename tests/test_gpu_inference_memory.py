"""Inference with fused activations and statistics: a call that no backward call can follow keeps no columns, with Parameters for
weights too, under no_grad and inference_mode."""
import ctypes

import pytest
import torch
import torch.nn as nn

from d2conv3d_amd import _lib, _ops, modules, util

pytestmark = pytest.mark.gpu

C, DIMS = 128, (8, 30, 53)


def _columns_bytes(dtype):
    desc = _lib.Conv3dDesc(1, C, C, *DIMS, 3, 3, 3, 1, 1, 1, 1, 1, 1, 1, 1, 1, 1, 1, *DIMS, _lib.D2C_F32 if dtype == torch.float32 else _lib.D2C_BF16,
                           _lib.D2C_F32, 0, 1.0, 7, 0)
    return _lib.load().d2c_conv3d_keep_bytes(ctypes.byref(desc), None)


def _peak(f):
    with torch.no_grad():
        f()                                       # (workspaces that stay)
    torch.cuda.synchronize()
    before = torch.cuda.memory_allocated()
    torch.cuda.reset_peak_memory_stats()
    f()
    torch.cuda.synchronize()
    return torch.cuda.max_memory_allocated() - before


@pytest.mark.parametrize("mode", [torch.no_grad, torch.inference_mode])
@pytest.mark.parametrize("form", ["offsets", "sized", "layer"])
@pytest.mark.parametrize("want_stats", [False, True])
def test_inference_keeps_no_columns(form, want_stats, mode, dev):
    g = torch.Generator(device=dev).manual_seed(1)
    rn = lambda *s: torch.randn(*s, generator=g, device=dev)
    x, m = rn(1, C, *DIMS).bfloat16(), torch.rand(1, 27, *DIMS, generator=g, device=dev)
    w, b = nn.Parameter((rn(C, C, 3, 3, 3) / (C * 27) ** 0.5).bfloat16()), nn.Parameter(rn(C).bfloat16())
    columns = _columns_bytes(torch.bfloat16)
    assert columns > 18 * x.numel() * 2
    if form == "offsets":
        off = rn(1, 81, *DIMS)
        call = lambda: _ops.deform_conv3d(x, off, m, w, b, 1, 1, 1, 1, 1, 1, 1, 1, 1, 1, 1, relu_scale=1.0, want_stats=want_stats)
    elif form == "sized":
        size = 0.5 + 2 * torch.rand(1, 3, *DIMS, generator=g, device=dev)
        call = lambda: _ops.deform_conv3d_sized(x, size, m, w, b, "xyz", "linear", 1, 1, 1, relu_scale=1.0, want_stats=want_stats)
    else:
        block = nn.Sequential(modules.MDConv3d(C, C, 3, padding=1, init="random"), nn.ReLU(), nn.GroupNorm(8, C)).to(dev, torch.bfloat16)
        holder = nn.ModuleList([block])
        (util.fuse_conv_act_norm if want_stats else util.fuse_output_activation)(holder)
        call = lambda: holder[0](x)

    def inference():
        with mode():
            call()
    # (deformation, output, statistics, workspaces: up to a few times the input)
    assert _peak(inference) < columns // 3
    # while a call that a backward call may follow keeps them
    assert _peak(call) > columns
