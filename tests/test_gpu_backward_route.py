"""Which kernels the products of the bfloat16 passes run on, at the edges of their tiles (the values are held elsewhere, where every kernel would do): the
grad-column rows (csrc/d2c_conv.hip, grad_col_kernel), grad_weight over columns (col_weight_kernel), the wide convolution kernel; and
the calls that stay on the kernels of the other shapes."""
import pytest
import torch

import d2conv3d_amd as d2c
from d2conv3d_amd import _lib, _ops

pytestmark = pytest.mark.gpu


def _names(fn, *ids):
    lib = _lib.load()
    torch.cuda.synchronize()
    lib.d2c_profile_reset()
    lib.d2c_profile_enable(1)
    try:
        fn()
        torch.cuda.synchronize()
    finally:
        lib.d2c_profile_enable(0)
    r = tuple(lib.d2c_profile_kernel_name(i).decode() for i in ids)
    lib.d2c_profile_reset()
    return r


def _step(dev, cin, cout, dims, k=(3, 3, 3), groups=1, N=1, wanted="all", **kw):
    g = torch.Generator(device=dev).manual_seed(cin + cout)
    K, p = k[0] * k[1] * k[2], [v // 2 for v in k]
    rn = lambda *s: torch.randn(*s, generator=g, device=dev)
    x, w = rn(N, cin, *dims).bfloat16(), rn(cout, cin // groups, *k).bfloat16() / (cin * K) ** 0.5
    off = rn(N, 3 * groups * K, *dims)
    for name, t in (("x", x), ("off", off), ("w", w)):
        t.requires_grad_(wanted == "all" or name == wanted)
    out = d2c.deform_conv3d(x, off, None, w, None, 1, p, 1, groups, groups, **kw)
    gout = rn(*out.shape).bfloat16()
    return lambda: out.backward(gout)


@pytest.mark.parametrize("cin,cout,dims,k,N", [
    (128, 64, (3, 13, 17), (3, 3, 3), 1), (128, 136, (4, 9, 16), (3, 3, 3), 2), (256, 264, (4, 20, 33), (3, 3, 3), 1),
    (256, 512, (9, 31, 35), (3, 3, 3), 1), (256, 192, (3, 12, 13), (1, 1, 5), 3), (512, 70, (2, 15, 31), (1, 3, 1), 1), (1024, 200, (7, 29, 31), (1, 5, 1), 1)])
def test_products_of_one_weight_group(cin, cout, dims, k, N, dev):
    assert _names(_step(dev, cin, cout, dims, k, N=N), _lib.PROF_BWD_DATA, _lib.PROF_BWD_WEIGHT) == ("grad_col_kernel", "col_weight_kernel")


@pytest.mark.parametrize("kw,data,weight", [
    # no room for the sums where the grad-column rows were: 14 and 81 blocks of 128 and 256 output channels x 1 KB, 0.7 and 8.6 MB of rows
    (dict(cin=128, cout=8, dims=(3, 5, 7)), "grad_col_kernel", "tiled_bwd_weight_col_kernel"),
    (dict(cin=256, cout=520, dims=(4, 12, 13)), "tiled_bwd_col32_kernel", "tiled_bwd_weight_col_kernel"),
    (dict(cin=256, cout=520, dims=(4, 24, 40)), "tiled_bwd_col32_kernel", "col_weight_kernel"),              # several passes
    (dict(cin=256, cout=128, dims=(4, 12, 13), groups=2), "tiled_bwd_col32_kernel", "tiled_bwd_weight_col_kernel"),
    (dict(cin=128, cout=72, dims=(4, 16, 17), wanted="w"), "", "tiled_bwd_weight_col_kernel"),               # kept columns, nothing else wanted
    (dict(cin=256, cout=128, dims=(4, 12, 13), backward_memory="in_place"), "tiled_bwd_col32_kernel", "tiled_bwd_weight_col_kernel"),
])
def test_products_of_other_calls(kw, data, weight, dev):
    before = _ops.config.keep_columns()
    if "backward_memory" in kw:
        _ops.config.set_keep_columns(False)
    try:
        assert _names(_step(dev, **kw), _lib.PROF_BWD_DATA, _lib.PROF_BWD_WEIGHT) == (data, weight)
    finally:
        _ops.config.set_keep_columns(before["on"], before["max_bytes"])


@pytest.mark.parametrize("N,cout,dims", [(1, 256, (7, 120, 107)), (2, 200, (3, 121, 122)), (1, 129, (7, 121, 107)), (1, 256, (8, 96, 97)), (2, 200, (3, 41, 50))])
def test_wide_convolution(N, cout, dims, dev):
    x, w, one = torch.randn(N, 128, *dims, device=dev).bfloat16(), torch.randn(cout, 128, 3, 3, 3, device=dev).bfloat16(), (1, 1, 1)
    assert _names(lambda: _ops.plain_conv3d(x, w, None, one, one, one), _lib.PROF_FWD) == ("conv_wide_kernel",)
