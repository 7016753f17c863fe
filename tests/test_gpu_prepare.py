"""Float32 input and grad_input moved between their layouts in 64 x 64 tiles (csrc/d2c_tiled.hip, d2c_tiled_bwd.hip), where a tile ends
inside the channels or the positions, and next to it where vectors of four do not fit: the operator at zero offsets against the
plain convolution."""
import pytest
import torch
import torch.nn.functional as F

import d2conv3d_amd as d2c
from _util import rel_l2

pytestmark = pytest.mark.gpu


# (N, C, dims, groups): 256 tiles and more, positions of a sample a multiple of four or not
@pytest.mark.parametrize("N,C,dims,depthwise", [(2, 516, (2, 30, 17), True), (2, 516, (2, 31, 17), True), (1, 1028, (3, 20, 17), True),
                                                (3, 96, (6, 23, 30), False), (3, 96, (5, 27, 29), False)])
def test_layouts_in_large_tiles(N, C, dims, depthwise, dev):
    g = torch.Generator().manual_seed(C + dims[1])
    groups, O = (C, C) if depthwise else (1, 32)
    x = torch.randn(N, C, *dims, generator=g)
    w = torch.randn(O, C // groups, 3, 3, 3, generator=g) / (C // groups * 27) ** 0.5
    gout = torch.randn(N, O, *dims, generator=g)
    xr = x.double().requires_grad_(True)
    ref = F.conv3d(xr, w.double(), padding=1, groups=groups)
    ref.backward(gout.double())
    xd = x.to(dev).requires_grad_(True)
    out = d2c.deform_conv3d(xd, torch.zeros(N, 81, *dims, device=dev), None, w.to(dev), None, 1, 1, 1, groups, 1)
    out.backward(gout.to(dev))
    # (two-term operands of the products: up to 2^-16)
    assert rel_l2(out, ref) < 2e-5 and rel_l2(xd.grad, xr.grad) < 2e-5
