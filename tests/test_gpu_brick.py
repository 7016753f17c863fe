"""The kernels over sampling points sorted by 1x3x3 blocks of voxels, bfloat16: forward and all gradients against the CPU
oracle where a block, a product of 32 points, a set of channel chunks or the volume ends, with points on, across and beyond the
border; and the matrix products of the forward pass over sampled columns and of the grad-column rows at the edges of their tiles, at zero
offsets against the plain convolution."""
import pytest
import torch
import torch.nn.functional as F

import d2conv3d_amd as d2c
from oracle import cpu
from _util import out_dims, rel_l2

pytestmark = pytest.mark.gpu

# (N, Cin, Cout, dims, kernel, stride, dilation, G, mask)
CASES = {
    "one_voxel": (1, 64, 40, (1, 1, 1), (3, 3, 3), 1, 1, 1, True),
    "five_chunks": (2, 320, 40, (3, 7, 11), (3, 3, 3), 1, 1, 1, True),
    "two_groups_stride": (1, 128, 136, (5, 9, 10), (3, 3, 3), 2, 1, 2, True),
    "bar_without_mask": (1, 192, 64, (4, 5, 33), (1, 7, 1), 1, 1, 1, False),
    "nine_chunks_three_groups_dilated": (1, 576, 33, (2, 6, 8), (3, 3, 3), 1, 2, 3, True),
    "kept_columns_ragged": (1, 128, 72, (13, 31, 31), (3, 3, 3), 1, 1, 2, True),
    "columns_forward_ragged": (1, 256, 16, (1, 95, 131), (3, 3, 3), 1, 1, 1, True),
    # the smallest problems that sample columns: kept for the backward pass, in a forward call alone
    "kept_columns_two_chunks": (1, 128, 24, (2, 16, 33), (3, 3, 3), 1, 1, 1, True),
    "kept_columns_few_positions": (1, 512, 72, (1, 19, 22), (3, 3, 3), 1, 1, 2, True),
    "columns_forward_smallest": (1, 256, 130, (8, 32, 32), (3, 3, 3), 1, 1, 1, True),
    "columns_forward_many_chunks": (1, 576, 40, (1, 63, 66), (1, 7, 1), 1, 1, 1, False),
}


@pytest.mark.parametrize("name", list(CASES))
def test_sorted_points_against_the_oracle(name, dev):
    N, Cin, Cout, dims, ks, stride, dil, G, masked = CASES[name]
    pad = tuple(dil * (k // 2) for k in ks)
    od = out_dims(dims, ks, (stride,) * 3, pad, (dil,) * 3)
    K = ks[0] * ks[1] * ks[2]
    g = torch.Generator().manual_seed(len(name))
    x = torch.randn(N, Cin, *dims, generator=g).bfloat16()
    w = (torch.randn(Cout, Cin, *ks, generator=g) / (Cin * K) ** 0.5).bfloat16()
    b = torch.randn(Cout, generator=g).bfloat16()
    off = torch.randn(N, G * 3 * K, *od, generator=g) * 1.5
    flat = off.view(-1)
    flat[::7] = flat[::7].round()                     # on a voxel, some of them on the border
    flat[::11] *= 8                                   # far outside
    m = torch.sigmoid(torch.randn(N, G * K, *od, generator=g)) if masked else None
    gout = torch.randn(N, Cout, *od, generator=g).bfloat16()
    f = lambda t: t.float() if t is not None else None
    exp = cpu.conv3d_forward(f(x), off, m, f(w), f(b), stride, pad, dil, 1, G)
    eg = cpu.conv3d_backward(f(gout), f(x), off, m, f(w), True, stride, pad, dil, 1, G)
    ts = [t.to(dev) if t is not None else None for t in (x, off, m, w, b)]
    assert rel_l2(d2c.deform_conv3d(*ts, stride, pad, dil, 1, G), exp) < 1e-2
    ts = [t.requires_grad_(True) if t is not None else None for t in ts]
    out = d2c.deform_conv3d(*ts, stride, pad, dil, 1, G)
    out.backward(gout.to(dev))
    assert rel_l2(out, exp) < 1e-2
    for what, t, e in zip(("grad_input", "grad_offset", "grad_mask", "grad_weight", "grad_bias"), ts, eg):
        if t is not None:
            assert rel_l2(t.grad, e) < 2e-2, (what, rel_l2(t.grad, e))


@pytest.mark.parametrize("Cin,Cout,dims", [(256, 130, (13, 31, 31)), (256, 300, (1, 111, 115)), (320, 72, (6, 45, 46)),
                                           (512, 257, (2, 80, 81))])
def test_columns_forward_at_tile_edges(Cin, Cout, dims, dev):
    g = torch.Generator().manual_seed(Cin + Cout)
    x = torch.randn(1, Cin, *dims, generator=g).bfloat16()
    w = (torch.randn(Cout, Cin, 3, 3, 3, generator=g) / (Cin * 27) ** 0.5).bfloat16()
    b = torch.randn(Cout, generator=g).bfloat16()
    out = d2c.deform_conv3d(x.to(dev), torch.zeros(1, 81, *dims, device=dev), None, w.to(dev), b.to(dev), 1, 1, 1, 1, 1)
    assert rel_l2(out, F.conv3d(x.float(), w.float(), b.float(), padding=1)) < 5e-3


# (reductions of one to four steps, last column tiles that are not full, one to eight ranges of column tiles, positions of a
# sample that are not a multiple of eight)
@pytest.mark.parametrize("N,Cin,Cout,dims", [(1, 256, 40, (1, 95, 131)), (2, 64, 72, (6, 61, 67)), (1, 256, 130, (13, 31, 32)),
                                             (1, 320, 256, (2, 63, 65)), (1, 1024, 64, (1, 61, 60)), (1, 1024, 200, (1, 62, 60))])
def test_grad_columns_at_tile_edges(N, Cin, Cout, dims, dev):
    g = torch.Generator().manual_seed(Cin + Cout)
    x = torch.randn(N, Cin, *dims, generator=g).bfloat16()
    w = (torch.randn(Cout, Cin, 3, 3, 3, generator=g) / (Cin * 27) ** 0.5).bfloat16()
    gout = torch.randn(N, Cout, *dims, generator=g).bfloat16()
    xr = x.float().requires_grad_(True)
    F.conv3d(xr, w.float(), padding=1).backward(gout.float())
    xd = x.to(dev).requires_grad_(True)
    d2c.deform_conv3d(xd, torch.zeros(N, 81, *dims, device=dev), None, w.to(dev), None, 1, 1, 1, 1, 1).backward(gout.to(dev))
    assert rel_l2(xd.grad, xr.grad) < 1e-2


def _one_tap(Cin, Cout, ks, dev):
    """Weights that hand channel 0 of the middle tap to output channel 0."""
    w = torch.zeros(Cout, Cin, *ks)
    w[0, 0, ks[0] // 2, ks[1] // 2, ks[2] // 2] = 1
    return w.bfloat16().to(dev)


def test_a_sample_is_interpolated_with_float32_weights(dev):
    """Neighbours r0 and -r1 sampled where they cancel but for 2^-17 (r0 + r1): float32 weights leave an error of about 2^-25,
    0.3 % of the value, and its rounding to bfloat16 0.2 %; weights of 16 or 17 bits leave 5 % and more."""
    N, C, O, dims, ks = 1, 256, 64, (9, 105, 14), (1, 3, 3)
    g = torch.Generator().manual_seed(3)
    x = torch.randn(N, C, *dims, generator=g).bfloat16()
    r = (1 + torch.rand(dims, generator=g)).bfloat16()
    pos = torch.arange(dims[2])
    x[0, 0] = r * (1 - 2 * (pos % 2))
    r0, r1 = r[..., :-1].double(), r[..., 1:].double()
    frac = torch.zeros(dims)
    frac[..., :-1] = (r0 / (r0 + r1) + 2.0 ** -17).float()
    frac = (frac + pos) - pos                         # (what float32 keeps of it at this position)
    off = torch.zeros(N, 27, *dims)
    off[0, 3 * 4 + 2] = frac
    out = d2c.deform_conv3d(x.to(dev), off.to(dev), None, _one_tap(C, O, ks, dev), None, 1, (0, 1, 1), 1, 1, 1)
    f = frac[..., :-1].double()
    want = ((1 - f) * r0 - f * r1) * (1 - 2 * (pos[:-1] % 2))
    assert rel_l2(out[0, 0, ..., :-1], want) < 1e-2


def test_grad_input_adds_float32_weights(dev):
    """Two points of opposite grad_out in the same cell, their fractions f and f + 2^-19: the differences +-2^-19 remain, exact
    in bfloat16."""
    N, C, O, dims, ks = 1, 64, 64, (4, 30, 14), (1, 3, 3)
    g = torch.Generator().manual_seed(4)
    x = torch.randn(N, C, *dims, generator=g).bfloat16().to(dev).requires_grad_(True)
    f = (torch.randint(2 ** 16, 2 ** 19, (*dims[:2], dims[2] // 2), generator=g) | 1).float() * 2.0 ** -20       # (a 20-bit fraction)
    off = torch.zeros(N, 27, *dims)
    off[0, 3 * 4 + 2, ..., 0::2] = f
    off[0, 3 * 4 + 2, ..., 1::2] = f + 2.0 ** -19 - 1
    gout = torch.zeros(N, O, *dims)
    gout[:, 0, ..., 0::2], gout[:, 0, ..., 1::2] = 1, -1
    out = d2c.deform_conv3d(x, off.to(dev), None, _one_tap(C, O, ks, dev), None, 1, (0, 1, 1), 1, 1, 1)
    out.backward(gout.bfloat16().to(dev))
    want = torch.full(dims, 2.0 ** -19)
    want[..., 1::2] *= -1
    assert torch.equal(x.grad[0, 0].float().cpu(), want)


# infinities and NaN reach what touches them and nothing else: as in the oracle, whatever shares a brick, a product of 32 points
# or a set of chunks with them.  (The same masks; values where they are finite.)
@pytest.mark.parametrize("what", ["input", "mask", "grad_out"])
@pytest.mark.parametrize("bad", [float("nan"), float("inf")])
@pytest.mark.parametrize("Cin,Cout,dims,G", [(128, 40, (13, 31, 31), 2), (320, 33, (3, 9, 11), 1)])
def test_infinities_and_nan_stay_where_they_are(Cin, Cout, dims, G, bad, what, dev):
    g = torch.Generator().manual_seed(11)
    x = torch.randn(1, Cin, *dims, generator=g).bfloat16()
    w = (torch.randn(Cout, Cin, 3, 3, 3, generator=g) / (Cin * 27) ** 0.5).bfloat16()
    off = torch.randn(1, G * 81, *dims, generator=g)
    m = torch.sigmoid(torch.randn(1, G * 27, *dims, generator=g))
    gout = torch.randn(1, Cout, *dims, generator=g).bfloat16()
    mid = tuple(d // 2 for d in dims)
    if what == "input":
        x[0, 3][0, 0, 0] = x[0, 70][mid] = x[0, Cin - 1][tuple(d - 1 for d in dims)] = bad
    elif what == "mask":
        m[0, 13][mid] = m[0, 13][1, 1, 1] = bad
    else:
        gout[0, 5][mid] = gout[0, 0][1, 1, 1] = bad
    for at in (mid, (1, 1, 1)):                       # (points outside the volume, where the oracle forms 0 * inf, are not meant)
        off[(0, slice(None)) + at] *= 0.1
    exp = cpu.conv3d_forward(x.float(), off, m, w.float(), None, 1, 1, 1, 1, G)
    eg = cpu.conv3d_backward(gout.float(), x.float(), off, m, w.float(), False, 1, 1, 1, 1, G)
    ts = [t.to(dev).requires_grad_(True) for t in (x, off, m, w)]
    out = d2c.deform_conv3d(*ts[:3], ts[3], None, 1, 1, 1, 1, G)
    out.backward(gout.to(dev))
    for name, t, e in zip(("out", "grad_input", "grad_offset", "grad_mask", "grad_weight"), [out] + [t.grad for t in ts], (exp,) + eg[:4]):
        t = t.detach().float().cpu()
        assert torch.equal(t.isfinite(), e.isfinite()), (name, int((~t.isfinite()).sum()), int((~e.isfinite()).sum()))
        ok = e.isfinite()
        if ok.any():
            assert rel_l2(t[ok], e[ok]) < 2e-2, name


def test_a_bad_voxel_stays_where_it_is_in_inference(dev):
    g = torch.Generator().manual_seed(12)
    dims = (1, 95, 131)
    x = torch.randn(1, 256, *dims, generator=g).bfloat16()
    w = (torch.randn(16, 256, 3, 3, 3, generator=g) / (256 * 27) ** 0.5).bfloat16()
    off = torch.randn(1, 81, *dims, generator=g)
    x[0, 200, 0, 50, 60] = float("nan")
    x[0, 0, 0, 94, 130] = float("inf")
    exp = cpu.conv3d_forward(x.float(), off, None, w.float(), None, 1, 1, 1, 1, 1)
    out = d2c.deform_conv3d(x.to(dev), off.to(dev), None, w.to(dev), None, 1, 1, 1, 1, 1).float().cpu()
    assert torch.equal(out.isfinite(), exp.isfinite())
    assert rel_l2(out[exp.isfinite()], exp[exp.isfinite()]) < 1e-2
