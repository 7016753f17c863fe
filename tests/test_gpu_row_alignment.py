"""Tensors whose rows start at any element: odd volumes, and storage that begins one element behind an aligned address.  The layout kernels
(input and grad_out to channels-last and to fragments, grad_input back) read and write such rows in 16-byte pieces, with ends
of their own, and pieces that span samples.

Expected: what the same call gives on aligned copies (the same arithmetic on the same values), whose own values the oracle's tests hold.  Sums are added
up in varying order (two calls on the same tensors differ in their last bits, float32 outputs included, where a tile's steps are shared out): a relative
2-norm of 1e-6 (float32) and 2^-8 (bfloat16, rounded once)."""
import pytest
import torch

import d2conv3d_amd as d2c
from d2conv3d_amd import _ops
from _util import rel_l2

pytestmark = pytest.mark.gpu


def _shifted(t):
    buf = torch.empty(t.numel() + 1, dtype=t.dtype, device=t.device)
    out = buf[1:].view(t.shape)
    out.copy_(t)
    return out


def _case(n, c, o, dims, dtype, dev):
    g = torch.Generator().manual_seed(sum(dims) * 10 + n)
    rnd = lambda *s: torch.randn(*s, generator=g).to(dtype).to(dev)
    return (rnd(n, c, *dims), rnd(n, 81, *dims), torch.sigmoid(rnd(n, 27, *dims).float()).to(dtype), rnd(o, c, 3, 3, 3) * 0.05, rnd(o)), rnd(n, o, *dims)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("n,c,o,dims", [
    (3, 64, 64, (1, 1, 3)),          # fewer positions than a vector, pieces over three samples
    (3, 64, 64, (3, 5, 7)),
    (2, 128, 64, (3, 9, 11)),
    (2, 256, 192, (4, 17, 23)),      # sorted points, columns, two samples of 1564 positions
    (1, 256, 256, (5, 31, 33)),
])
def test_rows_of_any_alignment(n, c, o, dims, dtype, dev):
    args, gout = _case(n, c, o, dims, dtype, dev)
    results = []
    for place in (torch.clone, _shifted):
        a = [place(v).requires_grad_(True) for v in args]
        out = d2c.deform_conv3d(*a, 1, 1, 1)
        results.append((out.detach(),) + torch.autograd.grad(out, a, place(gout)))
    for got, want in zip(results[1], results[0]):
        assert rel_l2(got, want.float()) <= (1e-6 if dtype == torch.float32 else 2.0 ** -8)


@pytest.mark.parametrize("n,c,o,dims", [(3, 64, 30, (3, 5, 7)), (1, 128, 108, (4, 17, 23)), (2, 64, 64, (1, 1, 3))])
def test_branch_convolution_rows_of_any_alignment(n, c, o, dims, dev):
    (x, _, _, w, b), gout = _case(n, c, o, dims, torch.bfloat16, dev)
    results = []
    for place in (torch.clone, _shifted):
        a = [place(v).requires_grad_(True) for v in (x, w, b)]
        out = _ops.plain_conv3d(*a, (1, 1, 1), (1, 1, 1), (1, 1, 1))
        results.append((out.detach(),) + torch.autograd.grad(out, a, place(gout)))
    want = torch.nn.functional.conv3d(x.double().cpu(), w.double().cpu(), b.double().cpu(), 1, 1)
    assert rel_l2(results[1][0].cpu(), want.float()) <= 2.0 ** -8
    for got, ref in zip(results[1], results[0]):
        assert rel_l2(got, ref.float()) <= 2.0 ** -8


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("n,c,dims", [
    (2, 3, (1, 1, 1)), (1, 5, (2, 3, 5)), (2, 3, (3, 33, 63)), (1, 2, (4, 7, 64)), (1, 3, (5, 9, 65)), (1, 2, (9, 34, 131)), (2, 2, (6, 32, 128)),
])
def test_depthwise_rows_of_any_alignment(n, c, dims, dtype, dev):
    """The plain channel-separated convolution: widths around its vectors and tiles.  Expected: torch's convolution in float64, of values that
    are rounded once (2^-8 in bfloat16; float32 sums of at most 27 products, of all positions for grad_weight: 1e-5 of the largest)."""
    from d2conv3d_amd.depthwise_conv import depthwise_separable_conv3d
    g = torch.Generator().manual_seed(dims[2])
    rnd = lambda *s: torch.randn(*s, generator=g).to(dtype).to(dev)
    args, gout = (rnd(n, c, *dims), rnd(c, 1, 3, 3, 3), rnd(c)), rnd(n, c, *dims)
    ref = [v.double().cpu().requires_grad_(True) for v in args]
    eo = torch.nn.functional.conv3d(*ref, 1, 1, 1, c)
    want = (eo.detach(),) + torch.autograd.grad(eo, ref, gout.double().cpu())
    for place in (torch.clone, _shifted):
        a = [place(v).requires_grad_(True) for v in args]
        out = depthwise_separable_conv3d(*a, 1, 1, 1)
        for got, w in zip((out.detach(),) + torch.autograd.grad(out, a, place(gout)), want):
            err = (got.double().cpu() - w).abs()
            assert (err <= 1e-5 * max(1.0, w.abs().max().item()) + (2.0 ** -8 * w.abs() if dtype == torch.bfloat16 else 0.0)).all()
