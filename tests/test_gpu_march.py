"""The plain depthwise convolution's marching kernels (3x3x3, unit stride and dilation, padding 1) at the edges of their
tiles (32 rows, 64 columns, ranges of planes): forward and all gradients against torch's convolution in float64."""
import pytest
import torch
import torch.nn.functional as F

from d2conv3d_amd.depthwise_conv import depthwise_separable_conv3d
from _util import rel_l2

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("n,c,dims", [(1, 1, (1, 1, 1)), (2, 3, (2, 31, 63)), (1, 2, (9, 33, 64)), (1, 2, (17, 32, 68)),
                                      (3, 5, (5, 65, 129)), (1, 600, (6, 3, 4))])
def test_march_kernels_at_tile_edges(n, c, dims, dtype, dev):
    g = torch.Generator().manual_seed(sum(dims) + c)
    x, gout = (torch.randn(n, c, *dims, generator=g).to(dtype) for _ in range(2))
    w, b = torch.randn(c, 1, 3, 3, 3, generator=g).to(dtype), torch.randn(c, generator=g).to(dtype)
    ref = [t.double().requires_grad_(True) for t in (x, w, b)]
    exp = F.conv3d(*ref, padding=1, groups=c)
    exp.backward(gout.double())
    ts = [t.to(dev).requires_grad_(True) for t in (x, w, b)]
    out = depthwise_separable_conv3d(*ts, 1, 1, 1)
    out.backward(gout.to(dev))
    tol = 1e-5 if dtype == torch.float32 else 1e-2
    assert rel_l2(out.double(), exp) < tol
    for name, t, r in zip(("grad_input", "grad_weight", "grad_bias"), ts, ref):
        assert rel_l2(t.grad.double(), r.grad) < tol, name
    # one gradient wanted at a time: the parts of the backward kernel that are left out
    for i in range(3):
        one = [t.to(dev).requires_grad_(j == i) for j, t in enumerate((x, w, b))]
        depthwise_separable_conv3d(*one, 1, 1, 1).backward(gout.to(dev))
        assert torch.equal(one[i].grad, ts[i].grad)
