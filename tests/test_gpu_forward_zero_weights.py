"""An infinity in a corner of weight zero, under a sampling point on a voxel plane or a modulation of exactly zero: it
reaches nothing in the forward pass of problems with many positions, or with many steps in all, whichever kernel serves them."""
import pytest
import torch

import d2conv3d_amd as d2c

pytestmark = pytest.mark.gpu


# 161 tiles of 64 positions with up to 128 output channels; 6 tiles of 216 (bfloat16) / 432 steps with more
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("cin,cout,dims", [(64, 64, (3, 41, 83)), (64, 100, (3, 41, 83)), (512, 192, (4, 9, 9))])
def test_infinities_of_weight_zero_reach_nothing(cin, cout, dims, dtype, dev):
    g = torch.Generator().manual_seed(cin + cout)
    x = torch.randn(1, cin, *dims, generator=g).to(dtype)
    w = (torch.rand(cout, cin, 3, 3, 3, generator=g) + 0.1).to(dtype)
    m = torch.rand(1, 27, *dims, generator=g) + 0.1
    m[torch.rand(m.shape, generator=g) < 0.3] = 0.0
    at = tuple(d // 2 for d in dims)
    x[(0, 5) + at] = float("inf")
    # offsets of zero: tap (i, j, l) of a position reads the voxel (i - 1, j - 1, l - 1) away from it, and no other
    out = d2c.deform_conv3d(x.to(dev), torch.zeros(1, 81, *dims, device=dev), m.to(dev), w.to(dev), None, 1, 1, 1, 1, 1)
    touched = torch.zeros(dims, dtype=torch.bool)
    for k in range(27):
        p = tuple(a + 1 - o for a, o in zip(at, (k // 9, k // 3 % 3, k % 3)))
        touched[p] = m[(0, k) + p] != 0
    assert 0 < touched.sum() < 27
    assert torch.equal((~out[0].isfinite()).cpu(), touched.expand(cout, *dims))
