"""The order of a wavefront's steps in the forward kernel of small problems (csrc/d2c_tiled_wave.hip): one step, two, many; taps that change from
step to step and chunks of one tap; offsets as they are stored in either type, with and without a mask, and lanes without a position.

Expected values: the CPU oracle.  float32: 1e-4 relative, 1e-5 absolute, as everywhere; bfloat16: output rounded once and columns rounded once, 2e-2 in
the 2-norm."""
import pytest
import torch

import d2conv3d_amd as d2c
from d2conv3d_amd import _lib
from oracle import cpu
from _util import assert_close, rel_l2

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype,aux", [(torch.float32, torch.float32), (torch.bfloat16, torch.float32), (torch.bfloat16, torch.bfloat16)])
@pytest.mark.parametrize("masked", [True, False])
@pytest.mark.parametrize("cin,k,G", [(64, (1, 1, 1), 1), (512, (1, 1, 1), 1), (1024, (1, 1, 1), 2), (128, (1, 3, 1), 2), (192, (3, 3, 3), 1)])
def test_every_order_of_steps(cin, k, G, masked, dtype, aux, dev):
    g = torch.Generator().manual_seed(cin + G)
    dims, cout, K = (1, 3, 11), 48, k[0] * k[1] * k[2]
    x, w = torch.randn(1, cin, *dims, generator=g).to(dtype), (torch.randn(cout, cin, *k, generator=g) / (cin * K) ** 0.5).to(dtype)
    b, off = torch.randn(cout, generator=g).to(dtype), (torch.randn(1, G * 3 * K, *dims, generator=g) * 1.5).to(aux)
    m = torch.sigmoid(torch.randn(1, G * K, *dims, generator=g)).to(aux) if masked else None
    p = [v // 2 for v in k]
    f = lambda t: None if t is None else t.float()
    exp = cpu.conv3d_forward(f(x), f(off), f(m), f(w), f(b), 1, p, 1, 1, G)
    ts = [None if t is None else t.to(dev) for t in (x, off, m, w, b)]
    lib = _lib.load()
    lib.d2c_profile_reset()
    lib.d2c_profile_enable(1)
    try:
        out = d2c.deform_conv3d(*ts, 1, p, 1, 1, G)
        torch.cuda.synchronize()
    finally:
        lib.d2c_profile_enable(0)
    name = lib.d2c_profile_kernel_name(_lib.PROF_FWD).decode()
    lib.d2c_profile_reset()
    assert name == "tiled_fwd_wave_kernel"
    if dtype == torch.float32:
        assert_close(out, exp, 1e-4, 1e-5, "forward")
    else:
        assert rel_l2(out, exp) < 2e-2
