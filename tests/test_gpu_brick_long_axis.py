"""Sorted points on an axis of several million voxels, where the quotient by the blocks' three voxels is more than a float holds: forward and
gradients of the last thousand positions against the CPU oracle on that end of the map alone.  Offsets along the axis are halves, so that
positions are the same numbers up there (floats are half a voxel apart) and in the oracle's map; grad_out is zero elsewhere, so that grad_weight and
grad_bias are the end's as well.  Columns, grad-column rows and results are each rounded to bfloat16 once: 1e-2 and 2e-2 in the 2-norm, as for short axes."""
import pytest
import torch

import d2conv3d_amd as d2c
from oracle import cpu
from _util import rel_l2

pytestmark = pytest.mark.gpu

LENGTH, END, EDGE = 6_400_000, 1024, 16      # (positions up to EDGE of the oracle's map miss what lies in front of it)


@pytest.mark.parametrize("axis", [1, 2])
def test_the_far_end_of_a_long_axis(axis, dev):
    g = torch.Generator().manual_seed(axis)
    dims, end, kernel, pad = [1, 1, 1], [1, 1, 1], [1, 1, 1], [0, 0, 0]
    dims[axis], end[axis], kernel[axis], pad[axis] = LENGTH, END, 3, 1
    C, O, K = 64, 64, 3
    x, w, b = torch.randn(1, C, *end, generator=g).bfloat16(), (torch.randn(O, C, *kernel, generator=g) / (C * K) ** 0.5).bfloat16(), torch.randn(O, generator=g).bfloat16()
    off = torch.rand(1, K, 3, END, generator=g) * 1.8 - 0.9
    off[:, :, axis] = torch.randint(-4, 5, (1, K, END), generator=g) / 2
    off = off.view(1, 3 * K, *end)
    m = torch.sigmoid(torch.randn(1, K, *end, generator=g))
    gout = torch.randn(1, O, *end, generator=g).bfloat16()
    gout.view(1, O, END)[..., :EDGE] = 0

    def long(t, fill):
        r = fill(1, t.shape[1], *dims)
        r.view(1, t.shape[1], LENGTH)[..., -END:] = t.to(dev).view(1, -1, END)
        return r

    def tail(t):
        return t.detach().reshape(1, t.shape[1], -1)[..., -(END - EDGE):].float().cpu()

    noise = lambda *s: torch.randn(*s, device=dev, dtype=torch.bfloat16)
    zeros = lambda dtype: lambda *s: torch.zeros(*s, device=dev, dtype=dtype)
    ts = [long(x, noise), long(off, zeros(torch.float32)), long(m, zeros(torch.float32)), w.to(dev), b.to(dev)]
    ts = [t.requires_grad_(True) for t in ts]
    out = d2c.deform_conv3d(*ts, 1, pad, 1)
    out.backward(long(gout, zeros(torch.bfloat16)))
    f = lambda t: t.float()
    exp = cpu.conv3d_forward(f(x), off, m, f(w), f(b), 1, pad, 1)
    eg = cpu.conv3d_backward(f(gout), f(x), off, m, f(w), True, 1, pad, 1)
    assert rel_l2(tail(out), tail(exp)) < 1e-2
    for what, t, e in zip(("grad_input", "grad_offset", "grad_mask"), ts, eg):
        assert rel_l2(tail(t.grad), tail(e)) < 2e-2, what
    for what, t, e in zip(("grad_weight", "grad_bias"), ts[3:], eg[3:]):
        assert rel_l2(t.grad, e) < 2e-2, what
