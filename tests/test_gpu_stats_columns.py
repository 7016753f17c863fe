"""Output statistics of a call that keeps its columns for the backward pass: the same sums, output and gradients as without
columns, from the smallest problems that keep them on; where gradients are not wanted nothing is kept."""
import pytest
import torch

from d2conv3d_amd import _ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype,Cin,Cout,dims", [(torch.bfloat16, 128, 40, (2, 16, 33)), (torch.bfloat16, 256, 130, (3, 13, 17)),
                                                 (torch.float32, 64, 72, (8, 19, 21)), (torch.float32, 64, 136, (4, 17, 20))])
def test_statistics_beside_kept_columns(dtype, Cin, Cout, dims, dev):
    g = torch.Generator().manual_seed(Cin + Cout)
    rn = lambda *s: torch.randn(*s, generator=g)
    x, w, b = rn(1, Cin, *dims).to(dtype), (rn(Cout, Cin, 3, 3, 3) / (Cin * 27) ** 0.5).to(dtype), rn(Cout).to(dtype)
    off, m, gout = rn(1, 81, *dims), torch.sigmoid(rn(1, 27, *dims)), rn(1, Cout, *dims).to(dtype)
    before = _ops.config.keep_columns()
    got = {}
    try:
        for keep in (True, False):
            _ops.config.set_keep_columns(keep)
            ts = [t.to(dev).requires_grad_(True) for t in (x, off, m, w, b)]
            out, stats = _ops.deform_conv3d(*ts, 1, 1, 1, 1, 1, 1, 1, 1, 1, 1, 1, relu_scale=1.5, want_stats=True)
            assert (out.grad_fn.saved_tensors[-1] is not None) == keep
            assert not stats.requires_grad
            out.backward(gout.to(dev))
            got[keep] = [out.detach(), stats] + [t.grad for t in ts]
    finally:
        _ops.config.set_keep_columns(before["on"], before["max_bytes"])
    out, stats = got[True][:2]
    o = out.double().flatten(2)
    # (sums of float32 over the positions)
    torch.testing.assert_close(stats.double(), torch.stack([o.sum(2), o.square().sum(2)], 2), rtol=1e-5, atol=1e-3)
    for a, e in zip(got[True], got[False]):
        a, e = a.double(), e.double()
        assert (a - e).norm() / e.norm() < (1e-2 if dtype == torch.bfloat16 else 1e-5)
    with torch.no_grad():
        ref, st = _ops.deform_conv3d(*[t.to(dev) for t in (x, off, m, w, b)], 1, 1, 1, 1, 1, 1, 1, 1, 1, 1, 1, relu_scale=1.5, want_stats=True)
    assert (ref.double() - out.double()).norm() / out.double().norm() < (1e-2 if dtype == torch.bfloat16 else 1e-5)
