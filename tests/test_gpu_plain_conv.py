"""The ordinary convolution of the deformation branches (csrc/d2c_conv.hip) against torch's convolution in float32 on
the CPU: edges of its tiles (rows, output columns, channel blocks of 64 / 128), shared-out steps, samples that end
inside a tile, strides, dilations, filter shapes, calls without bias."""
import pytest
import torch
import torch.nn.functional as F

from d2conv3d_amd import _ops
from _util import rel_l2

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("case", [
    # N, Cin, Cout, dims, kernel, stride, padding, dilation, bias
    (1, 64, 30, (3, 6, 7), (3, 3, 3), (1, 1, 1), (1, 1, 1), (1, 1, 1), True),       # one tile, most of it past the end
    (2, 128, 108, (4, 9, 11), (3, 3, 3), (1, 1, 1), (1, 1, 1), (1, 1, 1), True),    # a sample ends inside a tile
    (1, 192, 32, (2, 8, 8), (3, 3, 3), (1, 1, 1), (1, 1, 1), (1, 1, 1), False),     # exactly one tile, half a channel block
    (3, 64, 33, (2, 7, 9), (3, 3, 3), (1, 2, 2), (1, 1, 1), (1, 1, 1), True),       # stride: voxels no output reads
    (1, 64, 64, (5, 6, 7), (3, 3, 3), (1, 1, 1), (2, 2, 2), (2, 2, 2), True),       # dilation
    (1, 128, 81, (1, 5, 40), (1, 3, 5), (1, 1, 1), (0, 1, 2), (1, 1, 1), True),     # other filter shapes
    (1, 64, 4, (3, 4, 5), (1, 1, 1), (1, 1, 1), (0, 0, 0), (1, 1, 1), True),        # a pointwise filter
    (1, 64, 216, (4, 10, 13), (5, 5, 5), (1, 1, 1), (2, 2, 2), (1, 1, 1), True),    # more taps than a round of the finishing kernel
    (2, 512, 864, (3, 12, 17), (3, 3, 3), (1, 1, 1), (1, 1, 1), (1, 1, 1), True),   # several column tiles
    (1, 256, 128, (6, 40, 47), (3, 3, 3), (1, 1, 1), (1, 1, 1), (1, 1, 1), True),   # many tiles
])
def test_against_torch(case):
    N, Cin, Cout, dims, k, s, p, d, has_bias = case
    dev = torch.device("cuda:0")
    g = torch.Generator().manual_seed(5)
    x = torch.randn(N, Cin, *dims, generator=g).bfloat16()
    w = (torch.randn(Cout, Cin, *k, generator=g) / (Cin * k[0] * k[1] * k[2]) ** 0.5).bfloat16()
    b = torch.randn(Cout, generator=g).bfloat16() if has_bias else None
    ts = [t.to(dev).requires_grad_(True) if t is not None else None for t in (x, w, b)]
    assert _ops.plain_conv3d_supported(ts[0], ts[1], s, p, d)
    out = _ops.plain_conv3d(*ts, s, p, d)
    gout = torch.randn(out.shape, generator=g).bfloat16()
    out.backward(gout.to(dev))
    es = [t.float().requires_grad_(True) if t is not None else None for t in (x, w, b)]
    e = F.conv3d(*es, s, p, d)
    e.backward(gout.float())
    assert rel_l2(out, e.detach()) < 4e-3
    for name, t, f in zip(("x", "weight", "bias"), ts, es):
        if t is not None:
            assert rel_l2(t.grad, f.grad) < 4e-3, name


def test_unsupported_shapes_are_refused():
    dev = torch.device("cuda:0")
    x, w = torch.zeros(1, 48, 3, 4, 5, device=dev).bfloat16(), torch.zeros(8, 48, 3, 3, 3, device=dev).bfloat16()
    assert not _ops.plain_conv3d_supported(x, w, (1, 1, 1), (1, 1, 1), (1, 1, 1))
    with pytest.raises(RuntimeError, match="multiple of 64"):
        _ops._lib.check(_ops._lib.load().d2c_plain_conv3d_forward(
            _ops.ctypes.byref(_ops._plain_desc(x, w, (1, 1, 1), (1, 1, 1), (1, 1, 1))), _ops._ptr(x), _ops._ptr(w), None,
            _ops._ptr(x), None, 0, None, 0, _ops._stream(dev)), "plain_conv3d")
