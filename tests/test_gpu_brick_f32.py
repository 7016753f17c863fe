"""The gradients over sorted points in float32 (csrc/d2c_brick.hip): against the CPU oracle where a block, a product of 32
points, a set of channel chunks or the volume ends, with points on, across and beyond the border; what the operands' split into three terms leaves;
infinities, NaN and numbers that have no such split."""
import pytest
import torch

import d2conv3d_amd as d2c
from oracle import cpu
from _util import out_dims, rel_l2

pytestmark = pytest.mark.gpu

# (N, Cin, Cout, dims, kernel, stride, dilation, groups, G, mask): chunks of 32 channels, sets of up to four
CASES = {
    "one_voxel": (1, 32, 40, (1, 1, 1), (3, 3, 3), 1, 1, 1, 1, True),
    "five_chunks": (2, 160, 40, (3, 7, 11), (3, 3, 3), 1, 1, 1, 1, True),
    "two_groups_stride": (1, 64, 136, (5, 9, 10), (3, 3, 3), 2, 1, 1, 2, True),
    "bar_without_mask": (1, 96, 64, (4, 5, 33), (1, 7, 1), 1, 1, 1, 1, False),
    "nine_chunks_three_groups_dilated": (1, 864, 33, (2, 6, 8), (3, 3, 3), 1, 2, 1, 3, True),
    "two_weight_groups": (2, 128, 64, (4, 9, 13), (3, 3, 3), 1, 1, 2, 2, True),
    "ranges_of_planes": (1, 64, 16, (40, 6, 7), (3, 3, 3), 1, 1, 1, 1, True),
    # the smallest problems that keep the columns of the forward call
    "kept_columns_narrow": (1, 64, 24, (8, 19, 20), (3, 3, 3), 1, 1, 1, 1, True),
    "kept_columns_wide": (1, 64, 136, (4, 17, 18), (3, 3, 3), 1, 1, 1, 2, True),
    "two_passes_over_output_channels": (1, 64, 330, (6, 13, 14), (3, 3, 3), 1, 1, 1, 1, True),
    "widest_weight_group": (1, 64, 256, (3, 8, 9), (3, 3, 3), 1, 1, 1, 1, True),
}


@pytest.mark.parametrize("name", list(CASES))
def test_sorted_points_against_the_oracle(name, dev):
    N, Cin, Cout, dims, ks, stride, dil, groups, G, masked = CASES[name]
    pad = tuple(dil * (k // 2) for k in ks)
    od = out_dims(dims, ks, (stride,) * 3, pad, (dil,) * 3)
    K = ks[0] * ks[1] * ks[2]
    g = torch.Generator().manual_seed(len(name))
    x = torch.randn(N, Cin, *dims, generator=g)
    w = torch.randn(Cout, Cin // groups, *ks, generator=g) / (Cin // groups * K) ** 0.5
    b = torch.randn(Cout, generator=g)
    off = torch.randn(N, G * 3 * K, *od, generator=g) * 1.5
    flat = off.view(-1)
    flat[::7] = flat[::7].round()                     # on a voxel, some of them on the border
    flat[::11] *= 8                                   # far outside
    m = torch.sigmoid(torch.randn(N, G * K, *od, generator=g)) if masked else None
    gout = torch.randn(N, Cout, *od, generator=g)
    eg = cpu.conv3d_backward(gout, x, off, m, w, True, stride, pad, dil, groups, G)
    exp = cpu.conv3d_forward(x, off, m, w, b, stride, pad, dil, groups, G)
    ts = [t.to(dev).requires_grad_(True) if t is not None else None for t in (x, off, m, w, b)]
    out = d2c.deform_conv3d(*ts, stride, pad, dil, groups, G)
    out.backward(gout.to(dev))
    # (the product of the forward pass and the grad-column product take two-term operands, which leave up to 2^-17 of either
    # factor: 2^-16 = 1.5e-5)
    assert rel_l2(out, exp) < 2e-5
    for what, t, e in zip(("grad_input", "grad_offset", "grad_mask", "grad_weight", "grad_bias"), ts, eg):
        if t is not None:
            assert rel_l2(t.grad, e) < 2e-5, (what, rel_l2(t.grad, e))


def test_three_terms_hold_a_float(dev):
    """Rows of 16 significant bits, made exactly (one output channel, factors of 8 bits), and offsets of 10 fractional bits: what
    is left is the rounding of sums in float32, 2^-24 each, of which a gradient has up to about a hundred (6e-7 when they add
    up like errors of random sign; two terms per operand would leave 4e-6 and more)."""
    g = torch.Generator().manual_seed(2)
    dims = (4, 9, 13)
    x = torch.randn(1, 96, *dims, generator=g)
    w = torch.randn(32, 96, 3, 3, 3, generator=g).bfloat16().float()
    off = (torch.randn(1, 81, *dims, generator=g) * 1024).round() / 1024
    m = torch.sigmoid(torch.randn(1, 27, *dims, generator=g))
    gout = torch.zeros(1, 32, *dims)
    gout[:, 0] = torch.randn(1, *dims, generator=g).bfloat16().float()
    eg = cpu.conv3d_backward(gout.double(), x.double(), off.double(), m.double(), w.double(), False, 1, 1, 1, 1, 1)
    ts = [t.to(dev).requires_grad_(True) for t in (x, off, m, w)]
    d2c.deform_conv3d(*ts, None, 1, 1, 1, 1, 1).backward(gout.to(dev))
    for what, t, e in zip(("grad_input", "grad_offset", "grad_mask"), ts, eg):
        assert rel_l2(t.grad, e) < 6e-7, (what, rel_l2(t.grad, e))


@pytest.mark.parametrize("what", ["input", "mask", "grad_out"])
@pytest.mark.parametrize("bad", [float("nan"), float("inf"), -float("inf")])
@pytest.mark.parametrize("Cin,Cout,dims,G", [(64, 40, (5, 9, 11), 2), (160, 33, (3, 9, 11), 1)])
def test_infinities_and_nan_stay_where_they_are(Cin, Cout, dims, G, bad, what, dev):
    g = torch.Generator().manual_seed(11)
    x = torch.randn(1, Cin, *dims, generator=g)
    w = torch.randn(Cout, Cin, 3, 3, 3, generator=g) / (Cin * 27) ** 0.5
    off = torch.randn(1, G * 81, *dims, generator=g)
    m = torch.sigmoid(torch.randn(1, G * 27, *dims, generator=g))
    gout = torch.randn(1, Cout, *dims, generator=g)
    mid = tuple(d // 2 for d in dims)
    if what == "input":
        x[0, 3][0, 0, 0] = x[0, 40][mid] = x[0, Cin - 1][tuple(d - 1 for d in dims)] = bad
    elif what == "mask":
        m[0, 13][mid] = m[0, 13][1, 1, 1] = bad
    else:
        gout[0, 5][mid] = gout[0, 0][1, 1, 1] = bad
    for at in (mid, (1, 1, 1)):                       # (points outside the volume, where the oracle forms 0 * inf, are not meant)
        off[(0, slice(None)) + at] *= 0.1
    eg = cpu.conv3d_backward(gout, x, off, m, w, False, 1, 1, 1, 1, G)
    ts = [t.to(dev).requires_grad_(True) for t in (x, off, m, w)]
    d2c.deform_conv3d(*ts, None, 1, 1, 1, 1, G).backward(gout.to(dev))
    for name, t, e in zip(("grad_input", "grad_offset", "grad_mask"), ts, eg):
        t = t.grad.cpu()
        assert torch.equal(t.isfinite(), e.isfinite()), (name, int((~t.isfinite()).sum()), int((~e.isfinite()).sum()))
        ok = e.isfinite()
        assert rel_l2(t[ok], e[ok]) < 2e-5, name


@pytest.mark.parametrize("big", [3.395e38, -3.4e38])
def test_numbers_next_to_the_largest(big, dev):
    """Finite, but the first of three terms rounds to an infinity."""
    g = torch.Generator().manual_seed(13)
    dims = (3, 9, 11)
    x = torch.randn(1, 64, *dims, generator=g)
    x[0, 40, 1, 4, 5] = big
    w = torch.randn(16, 64, 3, 3, 3, generator=g) / (64 * 27) ** 0.5
    off = torch.randn(1, 81, *dims, generator=g)
    m = torch.sigmoid(torch.randn(1, 27, *dims, generator=g))
    gout = torch.randn(1, 16, *dims, generator=g) * 0.01
    eg = cpu.conv3d_backward(gout.double(), x.double(), off.double(), m.double(), w.double(), False, 1, 1, 1, 1, 1)
    ts = [t.to(dev).requires_grad_(True) for t in (x, off, m)]
    d2c.deform_conv3d(*ts, w.to(dev), None, 1, 1, 1, 1, 1).backward(gout.to(dev))
    for name, t, e in zip(("grad_input", "grad_offset", "grad_mask"), ts, eg):
        t = t.grad.cpu()
        assert t.isfinite().all(), name
        at = e.abs() > 1e30                           # (the points that touch it; rel_l2 of the others)
        for sel in (at, ~at):
            if sel.any():
                scale = float(e[sel].abs().max())
                assert rel_l2(t[sel].double() / scale, e[sel] / scale) < 2e-5, name
