"""grad_weight of small 1-D problems, whose rows of grad_out begin at any element: odd lengths, tensors that begin in the middle of a vector,
the last values of the last row."""
import pytest
import torch

import d2conv3d_amd as d2c
from oracle import cpu
from _util import rel_l2

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("first", [0, 1, 3])
@pytest.mark.parametrize("length", [1, 7, 8, 9, 31, 64, 333])
def test_rows_of_any_start(length, first, dtype, dev):
    N, cin, cout = 2, 64, 70
    g = torch.Generator().manual_seed(length)
    rn = lambda *s: torch.randn(*s, generator=g)
    x, w, b = rn(N, cin, length).to(dtype), (rn(cout, cin, 3) / (cin * 3) ** 0.5).to(dtype), rn(cout).to(dtype)
    off, m, gout = rn(N, 3, length) * 1.5, torch.sigmoid(rn(N, 3, length)), rn(N, cout, length).to(dtype)
    # (what stands in front of the tensor and behind it belongs to no result)
    buf = torch.full((first + gout.numel() + 8,), float("nan"), dtype=dtype, device=dev)
    go = buf[first:first + gout.numel()].view(gout.shape).copy_(gout)
    ts = [t.to(dev).requires_grad_(True) for t in (x, off, m, w, b)]
    grads = torch.autograd.grad(d2c.deform_conv1d(*ts, 1, 1, 1, 1, 1), ts, go)
    eg = cpu.conv1d_backward(gout.float(), x.float(), off, m, w.float(), True, 1, 1, 1, 1, 1)
    for n, a, e in zip(("grad_input", "grad_offset", "grad_mask", "grad_weight", "grad_bias"), grads, eg):
        assert rel_l2(a, e) < (1e-5 if dtype == torch.float32 else 2e-2), n
