"""The DMA-gather forward kernel on narrow weight groups: 65 to 128 output channels whose weights take 8 MB and more, or up to 128
with 1024 input channels and 27 taps, on 160 tiles and more, most of its output tile empty.  Expected values: the same call in two halves of its output channels, which the kernel of the small
problems serves (its own tests compare it with the oracle): sums of the same products, up to the order of their float32 additions."""
import pytest
import torch

import d2conv3d_amd as d2c
from d2conv3d_amd import _lib
from _util import rel_l2

pytestmark = pytest.mark.gpu

CIN, COUT, DIMS = 960, 96, (8, 36, 37)             # 10 MB of weights; 166 tiles of 64 positions and 32 over


def tensors(dev, K=27):
    g = torch.Generator(device=dev).manual_seed(3)
    rn = lambda *s: torch.randn(*s, generator=g, device=dev)
    return (rn(1, CIN, *DIMS), rn(1, 3 * K, *DIMS) * 1.5, torch.sigmoid(rn(1, K, *DIMS)), rn(COUT, CIN, 3, 3, 3) / (CIN * K) ** 0.5,
            rn(COUT), rn(1, COUT, *DIMS))


def forward_kernel(call):
    lib = _lib.load()
    lib.d2c_profile_reset()
    lib.d2c_profile_enable(1)
    try:
        out = call()
        torch.cuda.synchronize()
    finally:
        lib.d2c_profile_enable(0)
    name = lib.d2c_profile_kernel_name(_lib.PROF_FWD).decode()
    lib.d2c_profile_reset()
    return out, name


def test_training_step_and_statistics(dev):
    *ts, gout = tensors(dev)
    one = [t.clone().requires_grad_(True) for t in ts]
    (out, stats), name = forward_kernel(lambda: d2c.deform_conv3d(*one, 1, 1, 1, 1, 1, output_stats=True))
    assert name == "tiled_fwd_dma_kernel"
    out.backward(gout)
    halves, grads = [], []
    for h in (slice(0, 48), slice(48, 96)):
        part = [t.clone() for t in ts[:3]] + [ts[3][h].clone(), ts[4][h].clone()]
        part = [t.requires_grad_(True) for t in part]
        o, name = forward_kernel(lambda: d2c.deform_conv3d(*part, 1, 1, 1, 1, 1))
        assert name == "tiled_fwd_wave_kernel"
        o.backward(gout[:, h])
        halves.append(o.detach())
        grads.append([t.grad for t in part])
    assert rel_l2(out, torch.cat(halves, 1)) < 2e-6
    for i in range(3):
        assert rel_l2(one[i].grad, grads[0][i] + grads[1][i]) < 1e-5
    for i in (3, 4):
        assert rel_l2(one[i].grad, torch.cat([grads[0][i], grads[1][i]])) < 2e-6
    o = out.detach().double().flatten(2)
    assert rel_l2(stats, torch.stack([o.sum(2), o.square().sum(2)], 2)) < 1e-6


@pytest.mark.parametrize("axes", [6, 1, 7])        # four, two and eight corners of a sampling point
def test_inference(axes, dev):
    *ts, _ = tensors(dev)
    with torch.no_grad():
        out, name = forward_kernel(lambda: d2c.deform_conv3d(*ts, 1, 1, 1, 1, 1, offset_axes=axes))
        assert name == "tiled_fwd_dma_kernel"
        want = [d2c.deform_conv3d(*ts[:3], ts[3][h].contiguous(), ts[4][h].contiguous(), 1, 1, 1, 1, 1, offset_axes=axes)
                for h in (slice(0, 48), slice(48, 96))]
    assert rel_l2(out, torch.cat(want, 1)) < 2e-6


@pytest.mark.parametrize("cin,cout,kernel", [(576, 128, "tiled_fwd_wave_kernel"), (608, 128, "tiled_fwd_dma_kernel"),
                                             (992, 64, "tiled_fwd_wave_kernel"), (1024, 64, "tiled_fwd_dma_kernel")])
def test_line_between_the_kernels(cin, cout, kernel, dev):
    """Weights of 8 MB; 27 taps of 1024 channels."""
    x, off, m, w, b = tensors(dev)[:5]
    w = w.repeat(2, 2, 1, 1, 1)[:cout, :cin].contiguous()
    x = torch.cat([x, x], 1)[:, :cin].contiguous()
    with torch.no_grad():
        out, name = forward_kernel(lambda: d2c.deform_conv3d(x, off, m, w, None, 1, 1, 1, 1, 1))
        assert name == kernel
        want = [d2c.deform_conv3d(x, off, m, w[h].contiguous(), None, 1, 1, 1, 1, 1) for h in (slice(0, 32), slice(32, cout))]
    assert rel_l2(out, torch.cat(want, 1)) < 2e-6


@pytest.mark.parametrize("cin,dims,kernel", [(1376, (4, 51, 52), "tiled_fwd_dma_kernel"), (1344, (4, 51, 52), "tiled_fwd_wave_kernel"),
                                             (1376, (3, 60, 60), "tiled_fwd_wave_kernel"), (1376, (1, 102, 103), "tiled_fwd_wave_kernel")])
def test_thin_maps(cin, dims, kernel, dev):
    """A third of the taps of one plane, three quarters of three planes', four fifths of four planes' lie inside."""
    g = torch.Generator(device=dev).manual_seed(4)
    rn = lambda *s: torch.randn(*s, generator=g, device=dev)
    x, off, m, w = rn(1, cin, *dims), rn(1, 81, *dims) * 1.5, torch.sigmoid(rn(1, 27, *dims)), rn(128, cin, 3, 3, 3) / (cin * 27) ** 0.5
    with torch.no_grad():
        out, name = forward_kernel(lambda: d2c.deform_conv3d(x, off, m, w, None, 1, 1, 1, 1, 1))
        assert name == kernel
        want = []
        for h in (slice(0, 64), slice(64, 128)):
            o, name = forward_kernel(lambda: d2c.deform_conv3d(x, off, m, w[h].contiguous(), None, 1, 1, 1, 1, 1))
            assert name == "tiled_fwd_wave_kernel"
            want.append(o)
    assert rel_l2(out, torch.cat(want, 1)) < 2e-6
