"""The 1-D backward pass on both sides of the line between the kernels of small problems and the others."""
import pytest
import torch

import d2conv3d_amd as d2c
from d2conv3d_amd import _lib
from oracle import cpu
from _util import rel_l2

pytestmark = pytest.mark.gpu


# items of 32 positions, 32 input channels and a tap: 2560 for 512 -> 256 channels in float32, 5500 in two passes of 256 output channels, 2048 else
@pytest.mark.parametrize("cin,cout,length,dtype,small", [(512, 256, 1696, torch.float32, True), (512, 256, 1697, torch.float32, False),
                                                         (512, 320, 3648, torch.float32, True), (512, 320, 3649, torch.float32, False),
                                                         (512, 72, 1344, torch.float32, True), (512, 72, 1345, torch.float32, False),
                                                         (512, 320, 1344, torch.bfloat16, True), (512, 320, 1345, torch.bfloat16, False)])
def test_either_side_of_the_line(cin, cout, length, dtype, small, dev):
    g = torch.Generator().manual_seed(length)
    rn = lambda *s: torch.randn(*s, generator=g)
    x, w, b = rn(1, cin, length).to(dtype), (rn(cout, cin, 3) / (cin * 3) ** 0.5).to(dtype), rn(cout).to(dtype)
    off, m, gout = rn(1, 3, length) * 1.5, torch.sigmoid(rn(1, 3, length)), rn(1, cout, length).to(dtype)
    ts = [t.to(dev).requires_grad_(True) for t in (x, off, m, w, b)]
    out = d2c.deform_conv1d(*ts, 1, 1, 1, 1, 1)
    lib = _lib.load()
    lib.d2c_profile_reset()
    lib.d2c_profile_enable(1)
    try:
        out.backward(gout.to(dev))
        torch.cuda.synchronize()
    finally:
        lib.d2c_profile_enable(0)
    name = lib.d2c_profile_kernel_name(_lib.PROF_BWD_DATA).decode()
    lib.d2c_profile_reset()
    assert (name == "conv1d_data_kernel") == small, name
    eg = cpu.conv1d_backward(gout.float(), x.float(), off, m, w.float(), True, 1, 1, 1, 1, 1)
    for n, t, e in zip(("grad_input", "grad_offset", "grad_mask", "grad_weight", "grad_bias"), ts, eg):
        assert rel_l2(t.grad, e) < (1e-5 if dtype == torch.float32 else 2e-2), n
