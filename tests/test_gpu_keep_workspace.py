"""Workspace of a forward call that leaves input, sampling points and columns in the caller's buffer: the operands of the product and its
partial sums, no room for the input, and nothing written behind it."""
import ctypes

import pytest
import torch

from d2conv3d_amd import _lib
from _util import rel_l2

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,cin,cout,dims,G", [(2, 256, 40, (3, 13, 17), 1), (1, 256, 256, (8, 30, 54), 2), (1, 512, 304, (4, 17, 19), 8)])
def test_no_room_for_what_the_caller_holds(N, cin, cout, dims, G, dev):
    lib = _lib.load()
    g = torch.Generator(device=dev).manual_seed(cout)
    rn = lambda *s: torch.randn(*s, generator=g, device=dev)
    x, w, b = rn(N, cin, *dims).bfloat16(), (rn(cout, cin, 3, 3, 3) / (cin * 27) ** 0.5).bfloat16(), rn(cout).bfloat16()
    off, m = rn(N, G * 81, *dims) * 1.5, torch.sigmoid(rn(N, G * 27, *dims))
    desc = _lib.Conv3dDesc(N, cin, cout, *dims, 3, 3, 3, 1, 1, 1, 1, 1, 1, 1, 1, 1, 1, G, *dims, _lib.D2C_BF16, _lib.D2C_F32, 0, 1.0, 7, 0)
    d = ctypes.byref(desc)
    nb, least = lib.d2c_conv3d_forward_keep_workspace_bytes(d, None), lib.d2c_conv3d_forward_least_workspace_bytes(d, None)
    keep, columns = lib.d2c_conv3d_keep_bytes(d, None), lib.d2c_conv3d_columns_bytes(d, None)
    assert keep > 27 * x.numel() * 2
    # weights in tiles of up to 256 output channels, partial sums of the last round of 256 tiles: 64 - 256 positions x 256 channels each
    assert 0 < nb <= 27 * cin * ((cout + 255) // 256 * 256) * 2 + 256 * 256 * 256 * 4
    p = lambda t: ctypes.c_void_p(t.data_ptr())
    st = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    out = []
    for size in (nb, nb + x.numel() * 2):
        ws = torch.full((size + 4096,), 0xA5, dtype=torch.uint8, device=dev)
        buf = torch.full((keep + 4096,), 0xA5, dtype=torch.uint8, device=dev)
        o = torch.empty(N, cout, *dims, dtype=x.dtype, device=dev)
        _lib.check(lib.d2c_conv3d_forward_columns(d, None, p(x), p(off), p(m), p(w), p(b), p(o), p(buf), keep, p(ws), size, st), "forward")
        assert bool((ws[size:] == 0xA5).all()) and bool((buf[keep:] == 0xA5).all())
        out.append(o)
    ws, o = torch.empty(least, dtype=torch.uint8, device=dev), torch.empty_like(out[0])
    _lib.check(lib.d2c_conv3d_forward(d, p(x), p(off), p(m), p(w), p(b), p(o), p(ws), least, st), "gathering")
    assert rel_l2(out[0], o) < 4e-3 and rel_l2(out[1], o) < 4e-3


def test_headline_needs_no_second_input(dev):
    """2x512x8x30x54 in 8 offset groups: 14.2 MB of weights; the input alone takes 26.5."""
    desc = _lib.Conv3dDesc(2, 512, 512, 8, 30, 54, 3, 3, 3, 1, 1, 1, 1, 1, 1, 1, 1, 1, 1, 8, 8, 30, 54, _lib.D2C_BF16, _lib.D2C_F32, 0, 1.0, 7, 0)
    assert _lib.load().d2c_conv3d_forward_keep_workspace_bytes(ctypes.byref(desc), None) < 20e6
