"""The forward pass of narrow bfloat16 weight groups with offsets along one axis: the DMA-gather kernel on many tiles, with two corner rows
of a sampling point, the kernel whose wavefronts work alone below, right on both sides of the line."""
import pytest
import torch

import d2conv3d_amd as d2c
from d2conv3d_amd import _lib
from oracle import cpu
from _util import rel_l2

pytestmark = pytest.mark.gpu

DMA, WAVE = "tiled_fwd_dma_kernel", "tiled_fwd_wave_kernel"


# 384 tiles of 64 positions, 65 to 128 output channels
@pytest.mark.parametrize("cin,cout,dims,kernel", [(64, 65, (1, 143, 172), DMA), (64, 65, (1, 143, 171), WAVE), (128, 128, (3, 85, 97), DMA),
                                                  (64, 64, (1, 143, 172), WAVE)])
@pytest.mark.parametrize("axis", [0, 1, 2])
def test_one_axis(cin, cout, dims, kernel, axis, dev):
    g = torch.Generator().manual_seed(cin + cout)
    rn = lambda *s: torch.randn(*s, generator=g)
    x, w, b = rn(1, cin, *dims).bfloat16(), (rn(cout, cin, 1, 3, 1) / (cin * 3) ** 0.5).bfloat16(), rn(cout).bfloat16()
    off, m = rn(1, 9, *dims) * 1.5, torch.sigmoid(rn(1, 3, *dims))
    one = off.view(1, 3, 3, *dims).clone()
    one[:, :, [a for a in range(3) if a != axis]] = 0.0
    lib = _lib.load()
    with torch.no_grad():
        lib.d2c_profile_reset()
        lib.d2c_profile_enable(1)
        try:
            out = d2c.deform_conv3d(*(t.to(dev) for t in (x, off, m, w, b)), 1, (0, 1, 0), 1, 1, 1, offset_axes=1 << axis)
            torch.cuda.synchronize()
        finally:
            lib.d2c_profile_enable(0)
        name = lib.d2c_profile_kernel_name(_lib.PROF_FWD).decode()
        lib.d2c_profile_reset()
    assert name == kernel
    want = cpu.conv3d_forward(x.float(), one.view_as(off), m, w.float(), b.float(), (1, 1, 1), (0, 1, 0), (1, 1, 1), 1, 1)
    # (interpolated values and the output are rounded to bfloat16, 2^-9 each)
    assert rel_l2(out, want) < 4e-3
