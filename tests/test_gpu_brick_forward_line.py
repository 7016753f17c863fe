"""The forward pass of bfloat16 problems that keep nothing: over columns of sorted points from some positions on, gathering below, the
same results on either side of the line."""
import ctypes

import pytest
import torch

import d2conv3d_amd as d2c
from d2conv3d_amd import _lib
from _util import rel_l2

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("cin,cout,G,dims,columns", [(512, 136, 1, (5, 16, 32), True), (512, 136, 1, (3, 3, 284), False),
                                                     (512, 160, 2, (5, 16, 33), True), (256, 130, 1, (8, 20, 32), True),
                                                     (256, 130, 1, (1, 1, 5119), False), (192, 192, 1, (3, 37, 62), True)])
def test_either_side_of_the_line(cin, cout, G, dims, columns, dev):
    lib = _lib.load()
    desc = _lib.Conv3dDesc(1, cin, cout, *dims, 3, 3, 3, 1, 1, 1, 1, 1, 1, 1, 1, 1, 1, G, *dims, _lib.D2C_BF16, _lib.D2C_F32, 0, 1.0, 7, 0)
    d = ctypes.byref(desc)
    full, least = lib.d2c_conv3d_forward_workspace_bytes(d), lib.d2c_conv3d_forward_least_workspace_bytes(d, None)
    g = torch.Generator(device=dev).manual_seed(cout)
    rn = lambda *s: torch.randn(*s, generator=g, device=dev)
    x, w, b = rn(1, cin, *dims).bfloat16(), (rn(cout, cin, 3, 3, 3) / (cin * 27) ** 0.5).bfloat16(), rn(cout).bfloat16()
    off, m = rn(1, G * 81, *dims) * 1.5, torch.sigmoid(rn(1, G * 27, *dims))
    assert (full - least > 20 * x.numel() * 2) == columns
    with torch.no_grad():
        out = d2c.deform_conv3d(x, off, m, w, b, 1, 1, 1, 1, G)
    ws, want = torch.empty(least, dtype=torch.uint8, device=dev), torch.empty_like(out)
    p = lambda t: ctypes.c_void_p(t.data_ptr())
    st = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    _lib.check(lib.d2c_conv3d_forward(d, p(x), p(off), p(m), p(w), p(b), p(want), p(ws), least, st), "gathering")
    # (interpolated values are rounded to bfloat16, 2^-9 each, on both ways; the output once more)
    assert rel_l2(out, want) < 4e-3
