"""How the convolution kernel of large problems stores its tiles (csrc/d2c_conv.hip, conv_wide_kernel): four rows at a time where
rows come in fours, one by one otherwise, partial sums of shared-out tiles; with rows, columns and samples that end inside
a tile, and outputs that start off the alignment.  Against torch's convolution in float32 on the CPU; both round the same
sum to bfloat16 once, and the order of a float32 sum moves at most one rounding in a few hundred by 2^-8: 2e-3 in the 2-norm."""
import ctypes

import pytest
import torch
import torch.nn.functional as F

from d2conv3d_amd import _ops
from _util import rel_l2

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,cout,dims", [
    (1, 256, (7, 120, 107)),     # whole tiles, rows in fours
    (2, 200, (3, 121, 122)),     # ... an even number of rows that is no multiple of four, columns that end inside a tile
    (1, 129, (7, 121, 107)),     # ... an odd number
    (1, 256, (8, 96, 97)),       # whole tiles and shared-out ones
    (2, 200, (3, 41, 50)),       # shared-out ones
])
def test_tiles_are_stored_whole(N, cout, dims, dev):
    g = torch.Generator().manual_seed(cout)
    x = torch.randn(N, 128, *dims, generator=g).bfloat16()
    w = (torch.randn(cout, 128, 3, 3, 3, generator=g) / (128 * 27) ** 0.5).bfloat16()
    b = torch.randn(cout, generator=g).bfloat16()
    xd, wd, bd = x.to(dev), w.to(dev), b.to(dev)
    one = (1, 1, 1)
    lib, desc = _ops._lib.load(), _ops._plain_desc(xd, wd, one, one, one)
    size = N * cout * dims[0] * dims[1] * dims[2]
    out = torch.empty(size + 16, dtype=torch.bfloat16, device=dev)
    d = ctypes.byref(desc)
    ws = torch.empty(lib.d2c_plain_conv3d_forward_workspace_bytes(d), dtype=torch.uint8, device=dev)
    xcl = torch.empty(lib.d2c_plain_conv3d_input_bytes(d), dtype=torch.uint8, device=dev)
    e = F.conv3d(x.float(), w.float(), b.float(), 1, 1)
    for shift in (0, 1):         # `out` on 16 bytes, and two bytes behind
        out.fill_(7.0)
        at = out[8 + shift:8 + shift + size]
        _ops._lib.check(lib.d2c_plain_conv3d_forward(d, _ops._ptr(xd), _ops._ptr(wd), _ops._ptr(bd), _ops._ptr(at), _ops._ptr(xcl), xcl.numel(),
                                                     _ops._ptr(ws), ws.numel(), _ops._stream(dev)), "plain_conv3d")
        assert rel_l2(at.view(e.shape), e.bfloat16()) < 2e-3
        assert bool((out[:8 + shift] == 7).all()) and bool((out[8 + shift + size:] == 7).all())
