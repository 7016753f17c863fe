"""The backward pass of small 1-D problems (csrc/d2c_conv1d.hip) at the edges of its tiles (32 positions, 32 channels, 64
output channels, whole vectors of positions), against the CPU oracle to the tolerances of test_gpu_tiled.py; points on whole
positions, on the border and outside; gradients wanted one at a time."""
import pytest
import torch

import d2conv3d_amd as d2c
from oracle import cpu
from _util import assert_close, rel_l2

pytestmark = pytest.mark.gpu

# (N, Cin, Cout, L, k, stride, groups, G, mask)
CASES = {
    "one_position": (1, 64, 40, 1, 3, 1, 1, 1, True),
    "ragged": (3, 64, 65, 37, 3, 1, 1, 1, True),
    "vectors": (2, 128, 130, 48, 5, 1, 1, 2, True),
    "groups_stride": (2, 256, 192, 61, 3, 2, 2, 4, True),
    "wide_reduction_without_mask": (1, 64, 520, 33, 3, 1, 1, 1, False),
    "split_positions": (4, 64, 32, 255, 1, 1, 1, 1, True),
}


def tensors(name, dtype):
    N, cin, cout, L, k, stride, groups, G, masked = CASES[name]
    Lo = (L + 2 * (k // 2) - k) // stride + 1
    g = torch.Generator().manual_seed(len(name))
    bound = (cin // groups * k) ** -0.5
    x = torch.randn(N, cin, L, generator=g).to(dtype)
    w = ((torch.rand(cout, cin // groups, k, generator=g) * 2 - 1) * bound).to(dtype)
    b = ((torch.rand(cout, generator=g) * 2 - 1) * bound).to(dtype)
    off = torch.randn(N, G * k, Lo, generator=g) * 2
    flat = off.view(-1)
    flat[::5] = flat[::5].round()                     # on a position, some of them on the border
    flat[::11] *= 40                                  # far outside
    m = torch.sigmoid(torch.randn(N, G * k, Lo, generator=g)) if masked else None
    gout = torch.randn(N, cout, Lo, generator=g).to(dtype)
    return (x, off, m, w, b), gout, (stride, k // 2, 1, groups, G)


@pytest.mark.parametrize("aux", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("name", list(CASES))
def test_against_the_oracle(name, dtype, aux, dev):
    if dtype == torch.float32 and aux != dtype:
        pytest.skip("float32 problems have float32 offsets")
    (x, off, m, w, b), gout, geo = tensors(name, dtype)
    off, m = off.to(aux), m.to(aux) if m is not None else None
    f = lambda t: t.float() if t is not None else None
    eg = cpu.conv1d_backward(f(gout), f(x), f(off), f(m), f(w), True, *geo)
    ts = [t.to(dev).requires_grad_(True) if t is not None else None for t in (x, off, m, w, b)]
    d2c.deform_conv1d(*ts, *geo).backward(gout.to(dev))
    for what, t, e in zip(("grad_input", "grad_offset", "grad_mask", "grad_weight", "grad_bias"), ts, eg):
        if t is None:
            continue
        if dtype == torch.float32:
            assert_close(t.grad, e, 1e-4, 1e-5 * max(1.0, e.abs().max().item()), what)
        else:
            assert rel_l2(t.grad, e) < 2e-2, (what, rel_l2(t.grad, e))


@pytest.mark.parametrize("which", range(5))
def test_one_gradient_at_a_time(which, dev):
    (x, off, m, w, b), gout, geo = tensors("ragged", torch.float32)
    want = [t.to(dev).requires_grad_(True) for t in (x, off, m, w, b)]
    d2c.deform_conv1d(*want, *geo).backward(gout.to(dev))
    ts = [t.to(dev).requires_grad_(i == which) for i, t in enumerate((x, off, m, w, b))]
    d2c.deform_conv1d(*ts, *geo).backward(gout.to(dev))
    # (sums by atomics in another order)
    assert_close(ts[which].grad, want[which].grad, 1e-5, 1e-5 * max(1.0, want[which].grad.abs().max().item()), str(which))
