"""Channel-separated deformable convolution in bfloat16 on maps whose planes are too large for the descriptors of the forward kernel that requests rows
ahead (two rows and a voxel more than 2 GiB of channels-last input): its rows at either end against the same call on those rows alone, which that
kernel serves.  Offsets are sixteenths, so that both calls see the same fractions; the sums are the same, in the same order, and rounded once: one
unit in the last place (2^-8) for another contraction."""
import pytest
import torch

import d2conv3d_amd as d2c

pytestmark = pytest.mark.gpu


def test_forward_on_planes_of_two_gigabytes(dev):
    C, H, W, ROWS, EDGE = 1024, 1024, 1024, 48, 4
    assert (H * W + W + 2) * C * 2 >= 1 << 31 > (ROWS * W + W + 2) * C * 2
    g = torch.Generator(device=dev).manual_seed(5)
    x = torch.randn(1, C, 1, H, W, device=dev, dtype=torch.bfloat16, generator=g)
    off = (torch.randn(1, 3, 1, H, W, device=dev, generator=g) * 16).round().clamp(-48, 48) / 16
    off[:, 0] /= 4
    m = torch.rand(1, 1, 1, H, W, device=dev, generator=g)
    w, b = torch.randn(C, 1, 1, 1, 1, device=dev, generator=g).bfloat16(), torch.randn(C, device=dev, generator=g).bfloat16()
    out = d2c.deform_conv3d(x, off, m, w, b, 1, 0, 1, C)
    for rows, inner in ((slice(0, ROWS), slice(0, ROWS - EDGE)), (slice(H - ROWS, H), slice(EDGE, ROWS))):
        cut = [t[:, :, :, rows].contiguous() for t in (x, off, m)]
        want = d2c.deform_conv3d(*cut, w, b, 1, 0, 1, C)[:, :, :, inner].float()
        got = out[:, :, :, rows][:, :, :, inner].float()
        assert ((got - want).abs() <= 2.0 ** -8 * want.abs() + 1e-6).all()
