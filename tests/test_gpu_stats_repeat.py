"""Output statistics of narrow weight groups on large maps: summed in one order, so that repeated calls return the same bits."""
import pytest
import torch

import d2conv3d_amd as d2c

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("cin,cout", [(64, 64), (192, 100)])
def test_statistics_are_the_same_in_every_call(cin, cout, dtype, dev):
    dims = (8, 37, 61)                 # 282 tiles of 64 positions and 8 over, in two samples each
    g = torch.Generator(device=dev).manual_seed(cout)
    rn = lambda *s: torch.randn(*s, generator=g, device=dev)
    x, w, b = rn(2, cin, *dims).to(dtype), (rn(cout, cin, 3, 3, 3) / (cin * 27) ** 0.5).to(dtype), rn(cout).to(dtype)
    off, m = rn(2, 81, *dims), torch.sigmoid(rn(2, 27, *dims))
    with torch.no_grad():
        out, stats = d2c.deform_conv3d(x, off, m, w, b, 1, 1, 1, 1, 1, output_stats=True)
        for _ in range(4):
            o, s = d2c.deform_conv3d(x, off, m, w, b, 1, 1, 1, 1, 1, output_stats=True)
            assert torch.equal(o, out) and torch.equal(s, stats)
    o = out.double().flatten(2)
    # (float32 sums of 18056 values by 256 threads: 71 roundings in a thread's chain and 8 above it, each below 2^-24 of the sum of magnitudes)
    bound = 79 * 2.0 ** -24 * torch.stack([o.abs().sum(2), o.square().sum(2)], 2)
    assert bool(((stats.double() - torch.stack([o.sum(2), o.square().sum(2)], 2)).abs() <= bound).all())
