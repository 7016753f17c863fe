"""The forward pass of wide weight groups on a handful of position tiles with many steps each: the DMA-gather kernel, every work item cut into step
ranges, the kernel whose wavefronts work alone beside the lines, right on both sides."""
import pytest
import torch

import d2conv3d_amd as d2c
from d2conv3d_amd import _lib
from oracle import cpu
from _util import assert_close, rel_l2

pytestmark = pytest.mark.gpu

DMA, WAVE = "tiled_fwd_dma_kernel", "tiled_fwd_wave_kernel"


# four tiles of 64 positions; steps x samplings of 128 output channels at least 2560
@pytest.mark.parametrize("cin,cout,dims,groups,kernel", [(1024, 257, (1, 1, 193), 1, DMA), (1024, 257, (3, 8, 8), 1, WAVE), (1024, 256, (1, 1, 193), 1, WAVE),
                                                         (512, 769, (5, 9, 11), 1, DMA), (2048, 600, (1, 13, 17), 2, DMA), (2048, 600, (1, 12, 16), 2, WAVE)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_few_tiles(cin, cout, dims, groups, kernel, dtype, dev):
    cin *= 2 if dtype == torch.bfloat16 else 1         # (chunks of 64 channels, of 32 in float32)
    g = torch.Generator().manual_seed(cin + cout)
    rn = lambda *s: torch.randn(*s, generator=g)
    x, w, b = rn(1, cin, *dims).to(dtype), (rn(cout, cin // groups, 3, 3, 3) / (cin // groups * 27) ** 0.5).to(dtype), rn(cout).to(dtype)
    off, m = rn(1, groups * 81, *dims) * 1.5, torch.sigmoid(rn(1, groups * 27, *dims))
    lib = _lib.load()
    ts = [t.to(dev) for t in (x, off, m, w, b)]
    with torch.no_grad():
        lib.d2c_profile_reset()
        lib.d2c_profile_enable(1)
        try:
            out = d2c.deform_conv3d(*ts, 1, 1, 1, groups, groups)
            torch.cuda.synchronize()
        finally:
            lib.d2c_profile_enable(0)
        name = lib.d2c_profile_kernel_name(_lib.PROF_FWD).decode()
        lib.d2c_profile_reset()
    assert name == kernel
    one = (1, 1, 1)
    want = cpu.conv3d_forward(x.float(), off, m, w.float(), b.float(), one, one, one, groups, groups)
    if dtype == torch.float32:
        assert_close(out, want, 1e-4, 1e-5, name)
    else:
        # (interpolated values and the output are rounded to bfloat16, 2^-9 each)
        assert rel_l2(out, want) < 4e-3


# a hundred tiles of 64 positions, few steps: above 384 output channels the one, up to 384 the other; a hundred and some where the last round of work
# items is too short to be cut
@pytest.mark.parametrize("cin,cout,dims,k,kernel", [(64, 512, (4, 40, 40), 3, DMA), (64, 385, (1, 81, 79), 1, DMA), (64, 385, (1, 80, 79), 1, WAVE),
                                                    (64, 384, (4, 40, 40), 3, WAVE), (128, 520, (3, 65, 67), 3, DMA), (64, 130, (2, 68, 98), 1, DMA)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_few_steps_of_many_channels(cin, cout, dims, k, kernel, dtype, dev):
    g = torch.Generator().manual_seed(cin + cout)
    rn = lambda *s: torch.randn(*s, generator=g)
    x, w, b = rn(1, cin, *dims).to(dtype), (rn(cout, cin, k, 1, 1) / (cin * k) ** 0.5).to(dtype), rn(cout).to(dtype)
    off, m = rn(1, 3 * k, *dims) * 1.5, torch.sigmoid(rn(1, k, *dims))
    lib = _lib.load()
    with torch.no_grad():
        lib.d2c_profile_reset()
        lib.d2c_profile_enable(1)
        try:
            out = d2c.deform_conv3d(*(t.to(dev) for t in (x, off, m, w, b)), 1, (k // 2, 0, 0), 1, 1, 1)
            torch.cuda.synchronize()
        finally:
            lib.d2c_profile_enable(0)
        name = lib.d2c_profile_kernel_name(_lib.PROF_FWD).decode()
        lib.d2c_profile_reset()
    assert name == kernel
    want = cpu.conv3d_forward(x.float(), off, m, w.float(), b.float(), (1, 1, 1), (k // 2, 0, 0), (1, 1, 1), 1, 1)
    if dtype == torch.float32:
        assert_close(out, want, 1e-4, 1e-5, name)
    else:
        # (interpolated values and the output are rounded to bfloat16, 2^-9 each)
        assert rel_l2(out, want) < 4e-3
