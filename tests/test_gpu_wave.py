"""The forward kernel of small problems (csrc/d2c_tiled_wave.hip), whose wavefronts and workgroups share out the steps of a
tile of 32 positions, at the sizes where that can go wrong: tiles of one position and one past a tile's edge, fewer steps
than wavefronts, output channels around its tiles of 64 and 128, several weight groups, statistics of its output, columns.

Expected values: the CPU oracle, to the tolerances of test_gpu_tiled.py.  The partial sums are added in a fixed order, so
repeated calls give the same bits; a sum of all products over `terms` in another order differs by about
sqrt(terms) * 2^-24 of its scale, far below the 1e-4 of float32 checks."""
import ctypes

import pytest
import torch

import d2conv3d_amd as d2c
from d2conv3d_amd import _lib
from oracle import cpu
from _util import assert_close, rel_l2

pytestmark = pytest.mark.gpu

# (N, Cin, Cout, dims, kernel, groups, G)
CASES = {
    "one_position": (1, 64, 64, (1, 1, 1), (3, 3, 3), 1, 1),
    "tile_edge_33": (1, 64, 65, (1, 3, 11), (3, 3, 3), 1, 1),
    "one_step": (1, 64, 40, (2, 5, 7), (1, 1, 1), 1, 1),
    "samples_in_a_tile": (3, 64, 128, (1, 3, 5), (3, 3, 3), 1, 1),
    "many_splits": (1, 512, 64, (2, 4, 5), (3, 3, 3), 1, 1),
    "groups": (2, 256, 192, (2, 6, 7), (1, 3, 3), 2, 4),
    "wide": (1, 128, 300, (2, 5, 9), (3, 1, 1), 1, 2),
}


def tensors(case, dtype):
    N, cin, cout, dims, k, groups, G = case
    g = torch.Generator().manual_seed(77)
    K = k[0] * k[1] * k[2]
    bound = (cin // groups * K) ** -0.5
    x = torch.randn(N, cin, *dims, generator=g).to(dtype)
    w = ((torch.rand(cout, cin // groups, *k, generator=g) * 2 - 1) * bound).to(dtype)
    b = ((torch.rand(cout, generator=g) * 2 - 1) * bound).to(dtype)
    off = torch.randn(N, G * 3 * K, *dims, generator=g) * 1.5
    m = torch.sigmoid(torch.randn(N, G * K, *dims, generator=g))
    return x, off, m, w, b


def check(out, exp, dtype, what):
    if dtype == torch.float32:
        assert_close(out, exp, 1e-4, 1e-5, what)
    else:
        assert rel_l2(out, exp) < 2e-2, what


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("name", list(CASES))
def test_against_oracle(name, dtype, dev):
    case = CASES[name]
    N, cin, cout, dims, k, groups, G = case
    x, off, m, w, b = tensors(case, dtype)
    p = tuple(v // 2 for v in k)
    exp = cpu.conv3d_forward(x.float(), off, m, w.float(), b.float(), (1, 1, 1), p, (1, 1, 1), groups, G)
    ts = [t.to(dev) for t in (x, off, m, w, b)]
    out = d2c.deform_conv3d(*ts, 1, p, 1, groups, G)
    check(out, exp, dtype, name)
    for _ in range(4):
        assert torch.equal(d2c.deform_conv3d(*ts, 1, p, 1, groups, G), out)
    out2, stats = d2c.deform_conv3d(*ts, 1, p, 1, groups, G, output_stats=True)
    assert torch.equal(out2, out)
    o = out.float().flatten(2)
    assert_close(stats[..., 0], o.sum(2), 1e-5, 1e-5 * o.abs().sum(2).max().item(), "sum")
    assert_close(stats[..., 1], (o * o).sum(2), 1e-5, 1e-6, "sum of squares")


def test_without_room_for_partial_sums(dev):
    """A workspace that holds the operands alone: the steps of a tile stay with one workgroup."""
    lib = _lib.load()
    case = CASES["many_splits"]
    x, off, m, w, b = tensors(case, torch.float32)
    dims = case[3]
    desc = _lib.Conv3dDesc(1, 512, 64, *dims, 3, 3, 3, 1, 1, 1, 1, 1, 1, 1, 1, 1, 1, 1, *dims, _lib.D2C_F32, _lib.D2C_F32, 0, 1.0, 7, 0)
    d = ctypes.byref(desc)
    operands = (x.numel() * 4 + 256 + 255) // 256 * 256 + w.numel() * 4
    full = lib.d2c_conv3d_forward_workspace_bytes(d)
    assert operands < full
    exp = cpu.conv3d_forward(x, off, m, w, b, (1, 1, 1), (1, 1, 1), (1, 1, 1), 1, 1)
    ts = [t.to(dev) for t in (x, off, m, w, b)]
    p = lambda t: ctypes.c_void_p(t.data_ptr())
    for nb in (operands, full):
        ws = torch.empty(nb, dtype=torch.uint8, device=dev)
        out = torch.empty_like(exp, device=dev)
        st = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
        _lib.check(lib.d2c_conv3d_forward(d, *[p(t) for t in ts], p(out), p(ws), nb, st), "forward")
        assert_close(out, exp, 1e-4, 1e-5, f"{nb} bytes")


@pytest.mark.parametrize("cout", [64, 100])
def test_columns_of_narrow_weight_groups(cout, dev):
    """161 tiles of 64 positions, the last one with 29: the float32 training step keeps the columns of this kernel, and its
    grad_weight is a product over them (zeros past the last position)."""
    case = (1, 64, cout, (3, 41, 83), (3, 3, 3), 1, 1)
    x, off, m, w, b = tensors(case, torch.float32)
    gout = torch.randn(1, cout, *case[3], generator=torch.Generator().manual_seed(5))
    ts = [t.to(dev).requires_grad_(True) for t in (x, off, m, w, b)]
    out = d2c.deform_conv3d(*ts, 1, 1, 1, 1, 1)
    out.backward(gout.to(dev))
    one = (1, 1, 1)
    check(out, cpu.conv3d_forward(x, off, m, w, b, one, one, one, 1, 1), torch.float32, "forward")
    eg = cpu.conv3d_backward(gout, x, off, m, w, True, one, one, one, 1, 1)
    for n, t, e in zip(("grad_input", "grad_offset", "grad_mask", "grad_weight", "grad_bias"), ts, eg):
        assert_close(t.grad, e, 1e-4, 1e-5 * max(1.0, e.abs().max().item()), n)
