"""The forward pass of narrow weight groups with a few steps (taps x chunks of input channels): the DMA-gather kernel on many tiles, the kernel whose
eight wavefronts share out the steps of a tile beside the lines, right on both sides."""
import pytest
import torch

import d2conv3d_amd as d2c
from d2conv3d_amd import _lib
from oracle import cpu
from _util import assert_close, rel_l2

pytestmark = pytest.mark.gpu

DMA, WAVE = "tiled_fwd_dma_kernel", "tiled_fwd_wave_kernel"


# float32: chunks of 32 channels.  Above 64 output channels four steps and 384 tiles of 64 positions, twelve and 1600; below two and 1600
@pytest.mark.parametrize("cin,cout,dims,k,dtype,kernel", [(128, 65, (1, 143, 172), 1, torch.float32, DMA), (128, 65, (1, 143, 171), 1, torch.float32, WAVE),
                                                          (160, 65, (1, 143, 172), 1, torch.float32, WAVE), (64, 128, (2, 112, 112), 3, torch.bfloat16, DMA),
                                                          (128, 72, (8, 98, 131), 3, torch.float32, DMA), (192, 72, (8, 98, 130), 3, torch.bfloat16, WAVE),
                                                          (64, 64, (8, 98, 131), 1, torch.float32, DMA), (64, 40, (8, 98, 130), 1, torch.bfloat16, WAVE),
                                                          (96, 64, (8, 98, 131), 1, torch.float32, WAVE)])
def test_few_steps(cin, cout, dims, k, dtype, kernel, dev):
    g = torch.Generator().manual_seed(cin + cout)
    rn = lambda *s: torch.randn(*s, generator=g)
    x, w, b = rn(1, cin, *dims).to(dtype), (rn(cout, cin, 1, k, 1) / (cin * k) ** 0.5).to(dtype), rn(cout).to(dtype)
    off, m = rn(1, 3 * k, *dims) * 1.5, torch.sigmoid(rn(1, k, *dims))
    lib = _lib.load()
    with torch.no_grad():
        lib.d2c_profile_reset()
        lib.d2c_profile_enable(1)
        try:
            out = d2c.deform_conv3d(*(t.to(dev) for t in (x, off, m, w, b)), 1, (0, k // 2, 0), 1, 1, 1)
            torch.cuda.synchronize()
        finally:
            lib.d2c_profile_enable(0)
        name = lib.d2c_profile_kernel_name(_lib.PROF_FWD).decode()
        lib.d2c_profile_reset()
    assert name == kernel
    want = cpu.conv3d_forward(x.float(), off, m, w.float(), b.float(), (1, 1, 1), (0, k // 2, 0), (1, 1, 1), 1, 1)
    if dtype == torch.float32:
        assert_close(out, want, 1e-4, 1e-5, name)
    else:
        # (interpolated values and the output are rounded to bfloat16, 2^-9 each)
        assert rel_l2(out, want) < 4e-3
