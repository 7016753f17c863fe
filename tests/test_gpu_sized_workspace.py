"""d2c_conv3d_sized_forward with a workspace that holds its operands and no partial sums: accepted, like the same call of
d2c_conv3d_forward, and one byte less refused."""
import ctypes

import pytest
import torch

import d2conv3d_amd as d2c
from d2conv3d_amd import _lib
from d2conv3d_amd.grid import size_map_desc
from _util import rel_l2

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("cin,cout,dims", [(64, 64, (2, 5, 5)), (512, 64, (4, 14, 25)), (256, 128, (3, 17, 21))])
def test_the_operands_are_enough(cin, cout, dims, dtype, dev):
    lib = _lib.load()
    g = torch.Generator(device=dev).manual_seed(cin)
    rn = lambda *s: torch.randn(*s, generator=g, device=dev)
    x, w = rn(1, cin, *dims).to(dtype), (rn(cout, cin, 3, 3, 3) / (cin * 27) ** 0.5).to(dtype)
    size, m = 0.5 + 2 * torch.rand(1, 3, *dims, generator=g, device=dev), torch.rand(1, 27, *dims, generator=g, device=dev)
    dt = _lib.D2C_F32 if dtype == torch.float32 else _lib.D2C_BF16
    desc = _lib.Conv3dDesc(1, cin, cout, *dims, 3, 3, 3, 1, 1, 1, 1, 1, 1, 1, 1, 1, 1, 1, *dims, dt, _lib.D2C_F32, 0, 1.0)
    sdesc = size_map_desc(size, "xyz", (3, 3, 3), (1, 1, 1), "linear")
    d, s = ctypes.byref(desc), ctypes.byref(sdesc)
    # the input channels-last with 256 bytes of zeros, the weights
    up = lambda n: (n + 255) // 256 * 256
    operands = up(x.numel() * x.element_size() + 256) + up(w.numel() * w.element_size())
    full = lib.d2c_conv3d_sized_forward_workspace_bytes(d, s)
    assert operands < full
    want = d2c.deform_conv3d_sized(x, size, m, w, None, mode="xyz", padding=1)
    p = lambda t: ctypes.c_void_p(t.data_ptr())
    st = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    for nb in (operands, full):
        ws, out = torch.empty(nb, dtype=torch.uint8, device=dev), torch.empty_like(want)
        _lib.check(lib.d2c_conv3d_sized_forward(d, s, p(x), p(size), p(m), p(w), None, p(out), p(ws), nb, st), f"{nb} bytes")
        assert rel_l2(out, want) < (2e-6 if dtype == torch.float32 else 4e-3)
    assert lib.d2c_conv3d_sized_forward(d, s, p(x), p(size), p(m), p(w), None, p(out), p(ws), operands - 1, st) != 0
    assert "workspace" in _lib.last_error()
