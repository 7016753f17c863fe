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


@pytest.mark.parametrize("what", ["x", "grad_out"])
@pytest.mark.parametrize("bad", [float("nan"), float("inf")])
def test_a_bad_value_at_the_border_reaches_the_taps_that_meet_it(what, bad, dev):
    """grad_weight: the taps that pair the corner voxel, or the position at the corner, with something inside the volume (eight
    of 27), or a voxel in the first plane of another range of planes (all of them)."""
    g = torch.Generator().manual_seed(8)
    x, gout = (torch.randn(1, 3, 17, 33, 68, generator=g) for _ in range(2))
    t = x if what == "x" else gout
    t[0, 0, 0, 0, 0] = t[0, 2, 8, 5, 6] = bad
    w = torch.randn(3, 1, 3, 3, 3, generator=g)
    ts = [v.to(dev).requires_grad_(True) for v in (x, w)]
    depthwise_separable_conv3d(*ts, None, 1, 1, 1).backward(gout.to(dev))
    got = ts[1].grad.cpu()
    # (w[k] meets x[p + k - 1] and grad_out[p]: pairs with the corner need k >= 1 on every axis for a position, k <= 1 for a voxel)
    met = torch.zeros(3, 3, 3, dtype=torch.bool)
    met[(slice(0, 2),) * 3 if what == "x" else (slice(1, 3),) * 3] = True
    assert torch.equal(~got[0, 0].isfinite(), met)
    assert got[1].isfinite().all() and not got[2].isfinite().any()
    z = lambda v: torch.nan_to_num(v, 0.0, 0.0, 0.0)
    wr = w.double().requires_grad_(True)
    F.conv3d(z(x).double(), wr, padding=1, groups=3).backward(z(gout).double())
    assert rel_l2(got[0, 0][~met].double(), wr.grad[0, 0][~met]) < 1e-5 and rel_l2(got[1].double(), wr.grad[1]) < 1e-5
