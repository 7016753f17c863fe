"""The operators' calls in native code (csrc/torch/native.cpp) against the Python functions that they stand in for."""
import pytest
import torch

import d2conv3d_amd as d2c
from d2conv3d_amd import _ops
from d2conv3d_amd.depthwise_conv import depthwise_separable_conv3d
from _util import rel_l2

pytestmark = pytest.mark.gpu


def _rn(gen, *shape, dtype=torch.float32, std=1.0):
    return (torch.randn(*shape, generator=gen) * std).to(dtype)


# entry point -> (function of the tensors, the tensors of a seed)
def _conv3d(dtype=torch.float32):
    def tensors(seed):
        g = torch.Generator().manual_seed(seed)
        return [_rn(g, 1, 64, 3, 6, 7, dtype=dtype), _rn(g, 1, 81, 3, 6, 7, std=1.5), torch.sigmoid(_rn(g, 1, 27, 3, 6, 7)),
                _rn(g, 72, 64, 3, 3, 3, dtype=dtype, std=0.03), _rn(g, 72, dtype=dtype)]
    return lambda *t: d2c.deform_conv3d(*t, 1, 1, 1, 1, 1), tensors


def _sized():
    def tensors(seed):
        g = torch.Generator().manual_seed(seed)
        return [_rn(g, 1, 64, 3, 6, 7), torch.rand(1, 3, 3, 6, 7, generator=g) * 2 + 0.5, torch.sigmoid(_rn(g, 1, 27, 3, 6, 7)),
                _rn(g, 40, 64, 3, 3, 3, std=0.03), _rn(g, 40)]
    return lambda *t: d2c.deform_conv3d_sized(*t, mode="xyz", stride=1, padding=1, dilation=1), tensors


def _packed():
    def tensors(seed):
        g = torch.Generator().manual_seed(seed)
        return [_rn(g, 1, 64, 3, 6, 7), _rn(g, 1, 108, 3, 6, 7), _rn(g, 40, 64, 3, 3, 3, std=0.03), _rn(g, 40)]
    return lambda *t: _ops.deform_conv3d_packed(*t, 81, "sigmoid", (1, 1, 1), (1, 1, 1), (1, 1, 1), 1, 1), tensors


def _conv1d():
    def tensors(seed):
        g = torch.Generator().manual_seed(seed)
        return [_rn(g, 2, 64, 33), _rn(g, 2, 3, 33), torch.sigmoid(_rn(g, 2, 3, 33)), _rn(g, 48, 64, 3, std=0.1), _rn(g, 48)]
    return lambda *t: d2c.deform_conv1d(*t, 1, 1, 1, 1, 1), tensors


def _plain():
    def tensors(seed):
        g = torch.Generator().manual_seed(seed)
        return [_rn(g, 1, 64, 3, 6, 7, dtype=torch.bfloat16), _rn(g, 40, 64, 3, 3, 3, dtype=torch.bfloat16, std=0.03),
                _rn(g, 40, dtype=torch.bfloat16)]
    return lambda *t: _ops.plain_conv3d(*t, (1, 1, 1), (1, 1, 1), (1, 1, 1)), tensors


def _depthwise():
    def tensors(seed):
        g = torch.Generator().manual_seed(seed)
        return [_rn(g, 1, 64, 3, 6, 7), _rn(g, 64, 1, 3, 3, 3), _rn(g, 64)]
    return lambda *t: depthwise_separable_conv3d(*t, 1, 1, 1), tensors


ENTRIES = {"conv3d": _conv3d(), "conv3d_bf16": _conv3d(torch.bfloat16), "sized": _sized(), "packed": _packed(), "conv1d": _conv1d(),
           "plain": _plain(), "depthwise": _depthwise()}


def _on(dev, ts, grad=False):
    return [t.to(dev).requires_grad_(grad) for t in ts]


@pytest.mark.parametrize("name", list(ENTRIES))
def test_a_traced_call_is_the_call(name, dev):
    """torch.jit.trace of an entry point, replayed on other inputs: what the call returns for those, not memory that nothing
    has written."""
    fn, tensors = ENTRIES[name]
    with torch.no_grad():
        traced = torch.jit.trace(fn, tuple(_on(dev, tensors(1))), check_trace=False)
        for seed in (2, 3):
            ts = _on(dev, tensors(seed))
            want = fn(*ts)
            junk = torch.full((1 << 20,), float("nan"), device=dev)      # (what an allocation finds that nothing writes)
            del junk
            # (not bit for bit: float32 sums of shared-out steps are added with atomics)
            assert rel_l2(traced(*ts), want) < 1e-5, (name, seed)


@pytest.mark.parametrize("cls", ["MDConv3d", "XYZSizeConditionedMDConv3d"])
def test_a_traced_layer_is_the_layer(cls, dev):
    torch.manual_seed(5)
    layer = getattr(d2c, cls)(64, 40, 3, padding=1).to(dev)
    with torch.no_grad():
        layer.deform_params.weight.normal_(0, 0.03)
        x, y = (torch.randn(1, 64, 3, 6, 7, device=dev) for _ in range(2))
        traced = torch.jit.trace(layer, (x,), check_trace=False)
        want = layer(y)
        junk = torch.full((1 << 20,), float("nan"), device=dev)
        del junk
        assert rel_l2(traced(y), want) < 1e-5, cls
