"""Float32 training steps that keep no columns: which of the two ways of the backward pass the default takes, on both sides of the line,
and that both are right there."""
import ctypes

import pytest
import torch

import d2conv3d_amd as d2c
from d2conv3d_amd import _lib, _ops
from oracle import cpu
from _util import rel_l2

pytestmark = pytest.mark.gpu


# 27 taps x positions x (8 offset groups + 1) x passes of 256 output channels: 150000 lies between 617 and 618 positions of the first
@pytest.mark.parametrize("cin,cout,G,dims,columns", [(512, 128, 8, (1, 1, 617), False), (512, 128, 8, (2, 3, 103), True),
                                                     (256, 320, 1, (3, 20, 23), False), (256, 320, 1, (3, 20, 24), True),
                                                     (64, 320, 1, (3, 20, 24), False), (128, 200, 2, (4, 24, 24), False),
                                                     # several passes: sorted points from 128 positions on
                                                     (64, 320, 1, (4, 4, 8), False), (64, 320, 1, (1, 1, 127), True)])
def test_default_of_float32_problems_without_kept_columns(cin, cout, G, dims, columns, dev):
    lib = _lib.load()
    need = {}
    for flags in (_lib.BWD_GW_DEFAULT, _lib.BWD_GW_COLUMNS, _lib.BWD_GW_RESAMPLE):
        desc = _lib.Conv3dDesc(1, cin, cout, *dims, 3, 3, 3, 1, 1, 1, 1, 1, 1, 1, 1, 1, 1, G, *dims, _lib.D2C_F32, _lib.D2C_F32, 0, 1.0, 7, flags)
        need[flags] = lib.d2c_conv3d_backward_workspace_bytes(ctypes.byref(desc))
    assert need[_lib.BWD_GW_COLUMNS] > need[_lib.BWD_GW_RESAMPLE]
    assert need[_lib.BWD_GW_DEFAULT] == need[_lib.BWD_GW_COLUMNS if columns else _lib.BWD_GW_RESAMPLE]
    g = torch.Generator().manual_seed(cin + cout)
    rn = lambda *s: torch.randn(*s, generator=g)
    x, w, off = rn(1, cin, *dims), rn(cout, cin, 3, 3, 3) / (cin * 27) ** 0.5, rn(1, G * 81, *dims) * 1.5
    m, gout = torch.sigmoid(rn(1, G * 27, *dims)), rn(1, cout, *dims)
    eg = cpu.conv3d_backward(gout, x, off, m, w, False, 1, 1, 1, 1, G)
    before = _ops.config.keep_columns()
    _ops.config.set_keep_columns(False)
    try:
        for kw in (dict(), dict(backward_memory="columns"), dict(backward_memory="resample")):
            ts = [t.to(dev).requires_grad_(True) for t in (x, off, m, w)]
            d2c.deform_conv3d(*ts, None, 1, 1, 1, 1, G, **kw).backward(gout.to(dev))
            for t, e in zip(ts, eg):
                assert rel_l2(t.grad, e) < 1e-5, kw
    finally:
        _ops.config.set_keep_columns(before["on"], before["max_bytes"])


@pytest.mark.parametrize("wanted", ["all", "x+offset", "x+w", "w+offset"])
def test_calls_that_want_no_such_product_run_over_sorted_points(wanted, dev):
    """On the columns' side of the line: without grad_weight, or without grad_offset and grad_mask, nobody multiplies over columns."""
    cin, cout, G, dims = 512, 128, 8, (2, 3, 103)
    g = torch.Generator().manual_seed(8)
    rn = lambda *s: torch.randn(*s, generator=g)
    x, w, off = rn(1, cin, *dims), rn(cout, cin, 3, 3, 3) / (cin * 27) ** 0.5, rn(1, G * 81, *dims) * 1.5
    m, gout = torch.sigmoid(rn(1, G * 27, *dims)), rn(1, cout, *dims)
    eg = cpu.conv3d_backward(gout, x, off, m, w, False, 1, 1, 1, 1, G)
    need = {"all": (1, 1, 1, 1), "x+offset": (1, 1, 0, 0), "x+w": (1, 0, 0, 1), "w+offset": (0, 1, 0, 1)}[wanted]
    lib = _lib.load()
    before = _ops.config.keep_columns()
    _ops.config.set_keep_columns(False)
    try:
        ts = [t.to(dev).requires_grad_(bool(n)) for t, n in zip((x, off, m, w), need)]
        out = d2c.deform_conv3d(*ts, None, 1, 1, 1, 1, G)
        lib.d2c_profile_reset()
        lib.d2c_profile_enable(1)
        out.backward(gout.to(dev))
        torch.cuda.synchronize()
    finally:
        lib.d2c_profile_enable(0)
        _ops.config.set_keep_columns(before["on"], before["max_bytes"])
    name = lib.d2c_profile_kernel_name(_lib.PROF_BWD_AUX).decode()
    lib.d2c_profile_reset()
    assert name == ("aux_grad_kernel" if wanted in ("all", "w+offset") else "brick_grad_f32_kernel")
    for t, n, e in zip(ts, need, eg):
        if n:
            assert rel_l2(t.grad, e) < 1e-5
