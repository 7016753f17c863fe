"""Workspace of the bfloat16 backward pass over sorted points: what its products take shares places with what is written later, and a call runs
with as much as it did before grad_col_kernel served more than 256 output channels."""
import ctypes
import itertools

import pytest
import torch

from d2conv3d_amd import _lib
from oracle import cpu
from _util import rel_l2


def _desc(N, cin, cout, dims, k, G=1):
    p = [v // 2 for v in k]
    return _lib.Conv3dDesc(N, cin, cout, *dims, *k, 1, 1, 1, *p, 1, 1, 1, 1, G, *dims, _lib.D2C_BF16, _lib.D2C_F32, 0, 1.0, 7, 0)


@pytest.mark.parametrize("shape,most,most_kept", [
    ((2, 512, 512, (8, 30, 54), (3, 3, 3), 8), 1806.2e6, 928.5e6), ((2, 256, 256, (8, 30, 54), (3, 3, 3)), 825.3e6, 436.9e6),
    ((1, 256, 256, (32, 60, 108), (3, 3, 3)), 6502.4e6, 3395.1e6)])
def test_large_problems_need_no_more_than_they_did(shape, most, most_kept):
    lib, d = _lib.load(), ctypes.byref(_desc(*shape))
    assert lib.d2c_conv3d_backward_workspace_bytes(d) <= most
    assert lib.d2c_conv3d_backward_keep_workspace_bytes(d, None) <= most_kept


def _inputs(N, cin, cout, dims, k):
    g = torch.Generator().manual_seed(cin + cout)
    K = k[0] * k[1] * k[2]
    rn = lambda *s: torch.randn(*s, generator=g)
    x, w, b = rn(N, cin, *dims).bfloat16(), (rn(cout, cin, *k) / (cin * K) ** 0.5).bfloat16(), rn(cout).bfloat16()
    off, m, gout = rn(N, 3 * K, *dims) * 1.5, torch.sigmoid(rn(N, K, *dims)), rn(N, cout, *dims).bfloat16()
    eg = cpu.conv3d_backward(gout.float(), x.float(), off, m, w.float(), True, 1, [v // 2 for v in k], 1, 1, 1)
    return (x, off, m, w, b), gout, eg


def _ptr(t):
    return ctypes.c_void_p(t.data_ptr() if t is not None else 0)


def _stream():
    return ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)


@pytest.mark.gpu
@pytest.mark.parametrize("N,cin,cout,dims,k", [(2, 64, 512, (2, 13, 17), (1, 3, 1)), (1, 64, 260, (3, 9, 20), (1, 1, 3))])
def test_without_room_for_grad_out_behind_the_sums_per_point(N, cin, cout, dims, k, dev):
    """grad_out channels-last takes more than the 16 bytes a sampling point that it may have: without the rest the other kernel makes the
    grad-column rows, and one byte less than that is refused."""
    lib, desc = _lib.load(), _desc(N, cin, cout, dims, k)
    d, M, K = ctypes.byref(desc), N * dims[0] * dims[1] * dims[2], k[0] * k[1] * k[2]
    up = lambda n: (n + 255) // 256 * 256
    full = lib.d2c_conv3d_backward_workspace_bytes(d)
    least = full - (up(M * ((cout + 63) // 64 * 64) * 2 + 1024) - up(M * K * 16))
    assert least < full
    (x, off, m, w, b), gout, eg = _inputs(N, cin, cout, dims, k)
    t = [v.to(dev) for v in (gout, x, off, m, w)]
    names = []
    for size in (full, least):
        ws = torch.full((size + 4096,), 0xFF, dtype=torch.uint8, device=dev)
        r = [torch.empty_like(v) for v in t[1:]] + [torch.empty(cout, dtype=torch.bfloat16, device=dev)]
        lib.d2c_profile_reset()
        lib.d2c_profile_enable(1)
        try:
            rc = lib.d2c_conv3d_backward(d, *map(_ptr, t), *map(_ptr, r), _ptr(ws), size, _stream())
            torch.cuda.synchronize()
        finally:
            lib.d2c_profile_enable(0)
        _lib.check(rc, "backward")
        names.append(lib.d2c_profile_kernel_name(_lib.PROF_BWD_DATA).decode())
        lib.d2c_profile_reset()
        assert bool((ws[size:] == 0xFF).all())
        for a, e in zip(r, eg):
            assert rel_l2(a, e) < 2e-2
        assert lib.d2c_conv3d_backward(d, *map(_ptr, t), *map(_ptr, r), _ptr(ws), least - 1, _stream()) == 3
    assert names[0] == "grad_col_kernel" and names[1] != names[0]


@pytest.mark.gpu
@pytest.mark.parametrize("kept", [False, True])
def test_every_set_of_gradients_in_a_workspace_of_their_size(kept, dev):
    """grad_weight's sums lie where the grad-column rows do: with and without columns, alone and beside the others."""
    shape = (1, 128, 72, (4, 16, 17), (3, 3, 3))
    lib, desc = _lib.load(), _desc(*shape)
    d = ctypes.byref(desc)
    (x, off, m, w, b), gout, eg = _inputs(*shape)
    tx, toff, tm, tw, tb, tg = (v.to(dev) for v in (x, off, m, w, b, gout))
    if kept:
        keep, fw = lib.d2c_conv3d_keep_bytes(d, None), lib.d2c_conv3d_forward_keep_workspace_bytes(d, None)
        col, ws, out = torch.empty(keep, dtype=torch.uint8, device=dev), torch.empty(fw, dtype=torch.uint8, device=dev), torch.empty_like(tg)
        _lib.check(lib.d2c_conv3d_forward_columns(d, None, _ptr(tx), _ptr(toff), _ptr(tm), _ptr(tw), _ptr(tb), _ptr(out), _ptr(col), keep, _ptr(ws), fw,
                                                  _stream()), "forward")
    size = lib.d2c_conv3d_backward_keep_workspace_bytes(d, None) if kept else lib.d2c_conv3d_backward_workspace_bytes(d)
    for want in itertools.product((True, False), repeat=4):            # input, offset, mask, weight
        r = [torch.empty_like(v) if f else None for v, f in zip((tx, toff, tm, tw), want)] + [torch.empty_like(tb)]
        ws = torch.full((size + 4096,), 0xFF, dtype=torch.uint8, device=dev)
        if kept:
            rc = lib.d2c_conv3d_backward_columns(d, None, _ptr(tg), _ptr(tx), _ptr(toff), _ptr(tm), _ptr(tw), _ptr(col), keep, *map(_ptr, r), _ptr(ws), size,
                                                 _stream())
        else:
            rc = lib.d2c_conv3d_backward(d, _ptr(tg), _ptr(tx), _ptr(toff), _ptr(tm), _ptr(tw), *map(_ptr, r), _ptr(ws), size, _stream())
        _lib.check(rc, "backward")
        assert bool((ws[size:] == 0xFF).all()), want
        for a, e in zip(r, eg):
            assert a is None or rel_l2(a, e) < 2e-2, want
