"""The grad-column product of bfloat16 problems (csrc/d2c_conv.hip, grad_col_kernel): every number of 64-channel steps that its
registers hold, output channels that end inside one, rows that end inside a tile of 256, runs of workgroups that cross rows,
an odd number of (chunk, tap) pairs.

With all offsets zero and no modulation grad_input is the plain convolution's: sums of at most 27 rows, each rounded to
bfloat16 (2^-9 of an element at most, 1.2e-3 in the 2-norm), and one more rounding at the end: 3e-3 of float64."""
import pytest
import torch

import d2conv3d_amd as d2c
from _util import rel_l2

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,cin,cout,dims,k", [
    (1, 128, 8, (3, 5, 7), (3, 3, 3)),          # less than a tile of rows
    (1, 256, 40, (9, 31, 35), (3, 3, 3)),        # one step, not full; 39 row tiles of which the last has 37 rows
    (1, 256, 128, (9, 31, 35), (3, 3, 3)),       # two
    (2, 192, 136, (6, 33, 32), (3, 3, 3)),       # three, the last with 8 channels; 81 pairs; two samples, whole tiles
    (1, 256, 256, (9, 31, 35), (3, 3, 3)),       # four
    (1, 256, 264, (9, 31, 35), (3, 3, 3)),       # five
    (1, 256, 384, (9, 31, 35), (3, 3, 3)),       # six
    (1, 256, 400, (9, 31, 35), (3, 3, 3)),       # seven
    (1, 256, 512, (9, 31, 35), (3, 3, 3)),       # eight
    (3, 1024, 200, (7, 29, 31), (1, 5, 1)),      # 80 pairs of five taps
])
def test_zero_offsets_give_the_plain_gradient(N, cin, cout, dims, k, dev):
    g = torch.Generator().manual_seed(cin + cout)
    K, p = k[0] * k[1] * k[2], [v // 2 for v in k]
    x = torch.randn(N, cin, *dims, generator=g).bfloat16()
    w = (torch.randn(cout, cin, *k, generator=g) / (cin * K) ** 0.5).bfloat16()
    gout = torch.randn(N, cout, *dims, generator=g).bfloat16()
    e = torch.nn.grad.conv3d_input(x.shape, w.double(), gout.double(), 1, p)
    xd, wd = x.to(dev).requires_grad_(True), w.to(dev)
    off = torch.zeros(N, 3 * K, *dims, device=dev, requires_grad=True)
    d2c.deform_conv3d(xd, off, None, wd, None, 1, p, 1, 1, 1).backward(gout.to(dev))
    assert rel_l2(xd.grad, e) < 3e-3
