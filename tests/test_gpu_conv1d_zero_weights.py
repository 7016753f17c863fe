"""An infinity under a modulation of exactly zero, or next to a sampling point that lies on a position: it reaches no weight
gradient of the 1-D operator that it has no part in, whatever the size of the problem."""
import pytest
import torch

import d2conv3d_amd as d2c

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("cin,cout,length", [(64, 64, 100), (512, 320, 64), (64, 64, 20000)])
def test_infinities_of_weight_zero_reach_no_weight_gradient(cin, cout, length, dtype, dev):
    g = torch.Generator().manual_seed(cin + length)
    x = torch.randn(2, cin, length, generator=g)
    m = torch.rand(2, 3, length, generator=g) + 0.1
    gout = torch.rand(2, cout, length, generator=g) + 0.1
    at = length // 2
    x[0, 5, at] = float("inf")
    # offsets of zero: tap k of position p reads position p + k - 1 and no other
    m[0, 1, at] = m[0, 2, at - 1] = 0.0
    w = (torch.randn(cout, cin, 3, generator=g) * 0.02).to(dev, dtype).requires_grad_(True)
    off = torch.zeros(2, 3, length, device=dev).requires_grad_(True)
    out = d2c.deform_conv1d(x.to(dev, dtype), off, m.to(dev), w, None, 1, 1, 1, 1, 1)
    out.backward(gout.to(dev, dtype))
    bad = torch.zeros(cin, 3, dtype=torch.bool)
    bad[5, 0] = True
    assert torch.equal((~w.grad.isfinite()).cpu(), bad.expand(cout, cin, 3))
