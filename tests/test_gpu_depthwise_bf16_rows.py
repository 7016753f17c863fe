"""Channel-separated deformable convolution in bfloat16: its forward kernel requests the rows of a position ahead of their use, batches of 16 taps, tiles of 32
positions, slices of 256 channels.

Expected: the float32 call on the same values (another kernel, held to the oracle elsewhere); the output differs from it by one rounding, 2^-8 of an element, and
by the order of sums of 27 x 8 products, 1e-5 of the largest."""
import pytest
import torch

import d2conv3d_amd as d2c

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,c,og,dims,kernel", [
    (1, 4, 1, (1, 1, 1), (1, 1, 1)), (2, 64, 1, (2, 3, 5), (3, 3, 3)), (1, 260, 1, (3, 5, 7), (3, 3, 3)), (2, 512, 2, (4, 6, 9), (1, 3, 3)),
    (1, 256, 4, (4, 8, 8), (3, 3, 3)), (1, 64, 1, (2, 9, 17), (4, 4, 1)),
])
def test_forward_against_float32(n, c, og, dims, kernel, dev):
    g = torch.Generator().manual_seed(c + dims[2])
    k = kernel[0] * kernel[1] * kernel[2]
    pad = tuple(v // 2 for v in kernel)
    out_dims = [d + 2 * p - v + 1 for d, p, v in zip(dims, pad, kernel)]
    rnd = lambda *s: torch.randn(*s, generator=g).bfloat16().to(dev)
    args = (rnd(n, c, *dims), rnd(n, 3 * og * k, *out_dims) * 2, torch.sigmoid(rnd(n, og * k, *out_dims).float()).bfloat16(), rnd(c, 1, *kernel), rnd(c))
    out = d2c.deform_conv3d(*args, 1, pad, 1, c, og).float()
    want = d2c.deform_conv3d(*(v.float() for v in args), 1, pad, 1, c, og)
    assert ((out - want).abs() <= 2.0 ** -8 * want.abs() + 1e-5 * max(1.0, want.abs().max().item())).all()
