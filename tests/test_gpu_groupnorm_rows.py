"""Rows of the normalisation kernels: lengths at the edges of a vector, of a thread's vectors and of a workgroup's share, rows that start
at any element, few rows (several workgroups each) and many.

Expected: torch.nn.functional.group_norm and its gradients in float64.  Tolerances: an output is one fmaf of x with factors whose relative errors are
a few float32 roundings, of terms up to |x - mean| * rstd and |mean| * rstd; bfloat16 rounds it once more (2^-8).  grad_x has the group's sums beside it, divided by
the number of their terms: errors of a chain of additions stay below 1e-5 of the largest gradient."""
import pytest
import torch
import torch.nn.functional as F

from d2conv3d_amd import _ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("n,c,length", [
    (1, 4, 1), (1, 4, 7), (2, 4, 9), (1, 8, 1023), (1, 8, 8192), (1, 8, 8193), (1, 4, 40967), (1, 4, 65537), (2, 600, 8199),
])
def test_rows_against_torch(n, c, length, dtype, dev):
    g = torch.Generator().manual_seed(length)
    x = (torch.randn(n, c, length, generator=g) * 1.5 + 0.3).to(dtype)
    w, b = (torch.rand(c, generator=g) + 0.5).to(dtype), torch.randn(c, generator=g).to(dtype)
    gy = torch.randn(n, c, length, generator=g).to(dtype)
    xd, wd, bd = (v.to(dev).requires_grad_(True) for v in (x, w, b))
    y = _ops.group_norm_from_stats(xd, _ops.channel_stats(xd.detach()), wd, bd, 2, 1e-2)
    y.backward(gy.to(dev))
    xr, wr, br = (v.double().requires_grad_(True) for v in (x, w, b))
    ey = F.group_norm(xr, 2, wr, br, 1e-2)
    ey.backward(gy.double())
    ulp = 2.0 ** -8 if dtype == torch.bfloat16 else 0.0
    for got, want in ((y.detach(), ey.detach()), (xd.grad, xr.grad)):
        tol = 1e-5 * max(1.0, want.abs().max().item()) + ulp * want.abs()
        assert ((got.double().cpu() - want).abs() <= tol).all()
    for got, want, terms in ((wd.grad, wr.grad, (gy.double() * x.double()).abs().sum((0, 2))), (bd.grad, br.grad, gy.double().abs().sum((0, 2)))):
        assert ((got.double().cpu() - want).abs() <= 1e-5 * (1.0 + 4.0 * terms) + ulp * want.abs()).all()
