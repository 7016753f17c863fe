"""Float32 columns kept by the forward kernel of narrow weight groups while workgroups share out the steps of its tiles: the workspace
that such a call asks for has room for their partial sums, and output, columns (through grad_weight) and gradients are right."""
import ctypes

import pytest
import torch

import d2conv3d_amd as d2c
from d2conv3d_amd import _lib
from oracle import cpu
from _util import assert_close

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("cin,cout,dims", [(64, 64, (6, 17, 31)), (128, 100, (5, 25, 27)), (256, 72, (3, 15, 15))])     # 50, 53 and 11 tiles of 64 positions
def test_kept_columns_beside_partial_sums(cin, cout, dims, dev):
    g = torch.Generator().manual_seed(cout)
    rn = lambda *s: torch.randn(*s, generator=g)
    x, w, b, off = rn(1, cin, *dims), rn(cout, cin, 3, 3, 3) / (cin * 27) ** 0.5, rn(cout), rn(1, 81, *dims) * 1.5
    m, gout = torch.sigmoid(rn(1, 27, *dims)), rn(1, cout, *dims)
    desc = _lib.Conv3dDesc(1, cin, cout, *dims, 3, 3, 3, 1, 1, 1, 1, 1, 1, 1, 1, 1, 1, 1, *dims, _lib.D2C_F32, _lib.D2C_F32, 0, 1.0, 7, 0)
    lib, d = _lib.load(), ctypes.byref(desc)
    assert lib.d2c_conv3d_keep_bytes(d, None) > 0
    # the operands, and more: what the call without columns has
    up = lambda n: (n + 255) // 256 * 256
    operands = up(x.numel() * 4 + 256) + (cout + 63) // 64 * 64 * cin * 27 * 4
    assert lib.d2c_conv3d_forward_keep_workspace_bytes(d, None) == lib.d2c_conv3d_forward_workspace_bytes(d) > operands
    ts = [t.to(dev).requires_grad_(True) for t in (x, off, m, w, b)]
    out = d2c.deform_conv3d(*ts, 1, 1, 1, 1, 1)
    out.backward(gout.to(dev))
    one = (1, 1, 1)
    assert_close(out, cpu.conv3d_forward(x, off, m, w, b, one, one, one, 1, 1), 1e-4, 1e-5, "forward")
    eg = cpu.conv3d_backward(gout, x, off, m, w, True, one, one, one, 1, 1)
    for n, t, e in zip(("grad_input", "grad_offset", "grad_mask", "grad_weight", "grad_bias"), ts, eg):
        assert_close(t.grad, e, 1e-4, 1e-5 * max(1.0, e.abs().max().item()), n)
