"""Sums and sums of squares per channel of a long row, against float64: as exact as float32 sums of tiles of positions."""
import pytest
import torch

from d2conv3d_amd import _ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("P", [1, 7, 255, 257, 4095, 4104, 51360, 205440, 205441])
def test_against_float64(P, dtype, dev):
    g = torch.Generator(device=dev).manual_seed(P)
    x = (torch.randn(2, 24, P, generator=g, device=dev) + 1.0).to(dtype)
    stats = _ops.channel_stats(x)
    e = x.double()
    want = torch.stack([e.sum(2), e.square().sum(2)], 2)
    size = torch.stack([e.abs().sum(2), e.square().sum(2)], 2)
    # (a square, four additions in float32 and the result's own rounding, each below 2^-24 of the sum of magnitudes)
    assert bool(((stats.double() - want).abs() <= 6 * 2.0 ** -24 * size).all())
