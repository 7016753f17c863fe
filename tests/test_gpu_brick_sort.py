"""The sort of sampling points (csrc/d2c_brick.hip) where a workgroup's window does not hold all blocks of the volume, along z
and along x, so that points flung far enough are counted and filed outside of it; more taps than a workgroup takes; volumes
thinner than its tiles of positions.  Forward and all gradients against the CPU oracle, as in test_gpu_brick.py."""
import pytest

import test_gpu_brick as base

pytestmark = pytest.mark.gpu

CASES = {
    "window_of_planes": (1, 64, 16, (9, 60, 130), (3, 3, 3), 1, 1, 1, True),
    "window_along_x": (1, 64, 8, (7, 12, 720), (3, 3, 3), 1, 1, 1, False),
    "forty_nine_taps": (1, 64, 16, (2, 20, 23), (1, 7, 7), 1, 1, 1, True),
    "two_planes_strided": (2, 128, 16, (3, 18, 21), (3, 3, 3), 2, 1, 2, True),
}


@pytest.mark.parametrize("name", list(CASES))
def test_sorted_points_against_the_oracle(name, dev, monkeypatch):
    monkeypatch.setitem(base.CASES, name, CASES[name])
    base.test_sorted_points_against_the_oracle(name, dev)
