"""The marching kernels of the plain depthwise convolution (csrc/d2c_dwconv.hip) at rows of any width and alignment, tiles with
wavefronts below the volume, one and two tiles along x, ranges of planes that end inside the volume: forward and all gradients
against torch's convolution in float64 (float32: sums of 27 products and, for grad_weight, of all positions; bfloat16: the
rounding of the results)."""
import pytest
import torch
import torch.nn.functional as F

from d2conv3d_amd.depthwise_conv import depthwise_separable_conv3d
from _util import rel_l2

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("N,C,dims", [(1, 3, (1, 1, 1)), (2, 5, (3, 33, 5)), (1, 4, (9, 7, 63)), (1, 2, (17, 35, 64)), (2, 3, (5, 24, 65)),
                                      (1, 3, (4, 65, 66)), (1, 2, (2, 2, 131))])
def test_any_width(N, C, dims, dtype, dev):
    g = torch.Generator().manual_seed(sum(dims))
    x = torch.randn(N, C, *dims, generator=g).to(dtype)
    w = (torch.randn(C, 1, 3, 3, 3, generator=g) / 5).to(dtype)
    b = torch.randn(C, generator=g).to(dtype)
    gout = torch.randn(N, C, *dims, generator=g).to(dtype)
    e = [t.double().requires_grad_(True) for t in (x, w, b)]
    exp = F.conv3d(*e, padding=1, groups=C)
    exp.backward(gout.double())
    # tensors that begin on any element of a larger one
    hold = torch.empty(x.numel() + 1, dtype=dtype, device=dev)
    xd = hold[1:].view_as(x).copy_(x) if dims[2] % 2 else x.to(dev)
    ts = [xd.requires_grad_(True), w.to(dev).requires_grad_(True), b.to(dev).requires_grad_(True)]
    out = depthwise_separable_conv3d(*ts, (1, 1, 1), (1, 1, 1), (1, 1, 1))
    out.backward(gout.to(dev))
    tol = 1e-5 if dtype == torch.float32 else 4e-3
    for what, a, ex in zip(("out", "grad_input", "grad_weight", "grad_bias"), [out] + [t.grad for t in ts], [exp] + [t.grad for t in e]):
        assert rel_l2(a, ex) < tol, (what, rel_l2(a, ex))
