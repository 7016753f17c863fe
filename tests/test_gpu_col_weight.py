"""grad_weight of bfloat16 problems as a product over sampled columns (csrc/d2c_conv.hip, col_weight_kernel): tiles of output
channels and sets of four (chunk, tap) pairs that end early, positions that end inside a tile of 64 or 128, one and several
pieces, filters of few taps, a grad_weight off the alignment.

With all offsets zero and no modulation the columns are the input itself, so grad_weight is the plain convolution's: exact
products, float32 sums, one rounding to bfloat16 (2^-9 of an element at most, 1.2e-3 in the 2-norm): 2e-3 of float64."""
import ctypes

import pytest
import torch

import d2conv3d_amd as d2c
from d2conv3d_amd import _lib, _ops
from _util import rel_l2

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,cin,cout,dims,k", [
    (1, 128, 64, (3, 13, 17), (3, 3, 3)),        # 54 pairs; half a tile of output channels; 663 positions
    (1, 128, 128, (5, 11, 19), (3, 3, 3)),       # a whole tile; 1045 positions, an odd number of tiles of 64
    (2, 128, 136, (4, 9, 16), (3, 3, 3)),        # 136 of 256; whole tiles
    (1, 256, 264, (4, 20, 33), (3, 3, 3)),       # a second tile with 8 channels
    (3, 256, 192, (3, 12, 13), (1, 1, 5)),       # 20 pairs
    (1, 512, 70, (2, 15, 31), (1, 3, 1)),        # 24 pairs, output channels that end inside a block of 32
    (1, 128, 256, (8, 33, 40), (3, 3, 3)),       # several pieces
])
def test_zero_offsets_give_the_plain_gradient(N, cin, cout, dims, k, dev):
    g = torch.Generator().manual_seed(cin + cout)
    K, p = k[0] * k[1] * k[2], [v // 2 for v in k]
    x = torch.randn(N, cin, *dims, generator=g).bfloat16()
    w = (torch.randn(cout, cin, *k, generator=g) / (cin * K) ** 0.5).bfloat16()
    gout = torch.randn(N, cout, *dims, generator=g).bfloat16()
    e = torch.nn.grad.conv3d_weight(x.double(), w.shape, gout.double(), 1, p)
    xd, wd = x.to(dev).requires_grad_(True), w.to(dev).requires_grad_(True)
    off = torch.zeros(N, 3 * K, *dims, device=dev, requires_grad=True)
    d2c.deform_conv3d(xd, off, None, wd, None, 1, p, 1, 1, 1).backward(gout.to(dev))
    assert rel_l2(wd.grad, e) < 2e-3


def test_gradient_off_the_alignment(dev):
    g = torch.Generator().manual_seed(3)
    dims, cin, cout = (3, 14, 19), 128, 72
    x = torch.randn(1, cin, *dims, generator=g).bfloat16()
    w = (torch.randn(cout, cin, 3, 3, 3, generator=g) / (cin * 27) ** 0.5).bfloat16()
    gout = torch.randn(1, cout, *dims, generator=g).bfloat16()
    e = torch.nn.grad.conv3d_weight(x.double(), w.shape, gout.double(), 1, 1)
    desc = _lib.Conv3dDesc(1, cin, cout, *dims, 3, 3, 3, 1, 1, 1, 1, 1, 1, 1, 1, 1, 1, 1, *dims, _lib.D2C_BF16, _lib.D2C_F32, 0, 1.0, 7, 0)
    lib, d, ptr = _lib.load(), ctypes.byref(desc), _ops._ptr
    xd, wd, gd = x.to(dev), w.to(dev), gout.to(dev)
    off = torch.zeros(1, 81, *dims, device=dev)
    gx, goff = torch.empty_like(xd), torch.empty_like(off)
    ws = torch.empty(max(lib.d2c_conv3d_backward_workspace_bytes(d), 1), dtype=torch.uint8, device=dev)
    buf = torch.full((w.numel() + 16,), 7.0, dtype=torch.bfloat16, device=dev)
    gw = buf[9:9 + w.numel()]                  # two bytes behind a multiple of 16
    _lib.check(lib.d2c_conv3d_backward(d, ptr(gd), ptr(xd), ptr(off), None, ptr(wd), ptr(gx), ptr(goff), None, ptr(gw), None, ptr(ws), ws.numel(),
                                       _ops._stream(dev)), "backward")
    assert rel_l2(gw.view(w.shape), e) < 2e-3
    assert bool((buf[:9] == 7).all()) and bool((buf[9 + w.numel():] == 7).all())
