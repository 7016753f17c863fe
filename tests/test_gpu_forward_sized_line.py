"""The forward pass of narrow weight groups with offsets from a size map: the DMA-gather kernel where few chunks share a sampling point, the kernel
whose wavefronts work alone beside the lines, right on both sides."""
import pytest
import torch

import d2conv3d_amd as d2c
from d2conv3d_amd import _lib
from _util import rel_l2

pytestmark = pytest.mark.gpu

DMA, WAVE = "tiled_fwd_dma_kernel", "tiled_fwd_wave_kernel"
F32, BF16 = torch.float32, torch.bfloat16


# 64 channels a chunk in bfloat16, 32 in float32; 160 and 384 tiles of 64 positions
@pytest.mark.parametrize("cin,cout,dims,k,dtype,kernel", [(64, 65, (1, 101, 101), 3, BF16, DMA), (64, 65, (1, 101, 100), 3, BF16, WAVE),
                                                          (128, 72, (1, 143, 172), 3, BF16, DMA), (128, 72, (1, 143, 171), 3, BF16, WAVE),
                                                          (192, 72, (1, 143, 172), 3, BF16, WAVE), (64, 64, (1, 143, 172), 3, BF16, DMA),
                                                          (64, 64, (1, 143, 171), 3, BF16, WAVE), (64, 64, (1, 143, 172), 1, BF16, WAVE),
                                                          (64, 100, (1, 143, 172), 3, F32, DMA), (64, 64, (1, 143, 172), 3, F32, WAVE),
                                                          (96, 100, (1, 143, 172), 3, F32, WAVE), (64, 100, (1, 143, 171), 3, F32, WAVE)])
def test_either_side_of_the_lines(cin, cout, dims, k, dtype, kernel, dev):
    g = torch.Generator(device=dev).manual_seed(cin + cout)
    rn = lambda *s: torch.randn(*s, generator=g, device=dev)
    K = 3 * k
    x, w, b = rn(1, cin, *dims).to(dtype), (rn(cout, cin, 1, 3, k) / (cin * K) ** 0.5).to(dtype), rn(cout).to(dtype)
    size, m = 0.5 + 2 * torch.rand(1, 3, *dims, generator=g, device=dev), torch.rand(1, K, *dims, generator=g, device=dev)
    kw = dict(mode="xyz", padding=(0, 1, k // 2))
    lib = _lib.load()
    with torch.no_grad():
        lib.d2c_profile_reset()
        lib.d2c_profile_enable(1)
        try:
            out = d2c.deform_conv3d_sized(x, size, m, w, b, **kw)
            torch.cuda.synchronize()
        finally:
            lib.d2c_profile_enable(0)
        name = lib.d2c_profile_kernel_name(_lib.PROF_FWD).decode()
        lib.d2c_profile_reset()
        assert name == kernel
        off = d2c.offsets_from_size_map(size, "xyz", (1, 3, k), (1, 1, 1))
        want = d2c.deform_conv3d(x, off, m, w, b, 1, (0, 1, k // 2), 1, 1, 1)
    # (the same offsets; bfloat16: interpolated values and the output are rounded, 2^-9 each)
    assert rel_l2(out, want) < (1e-5 if dtype == F32 else 4e-3)
