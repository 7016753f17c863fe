"""The operators' calls in native code (csrc/torch/native.cpp) against the Python functions that they stand in for."""
import contextlib

import pytest
import torch

import d2conv3d_amd as d2c
from d2conv3d_amd import _ops, depthwise_conv
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


@pytest.fixture
def python_route():
    """A context in which every call goes through the Python functions."""
    @contextlib.contextmanager
    def route():
        with pytest.MonkeyPatch.context() as mp:
            mp.setattr(_ops, "_try_native", lambda *a: None)
            mp.setattr(depthwise_conv, "_try_native", lambda *a: None)
            yield
    return route


def _out_grad(out, seed=9):
    g = torch.Generator().manual_seed(seed)
    return torch.randn(*out.shape, generator=g).to(out)


def _plain_step(fn, ts, dev):
    out = fn(*ts)
    out.backward(_out_grad(out))
    return [out] + [t.grad for t in ts]


def _side_stream(fn, ts, dev):
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        out = fn(*ts)
        out.backward(_out_grad(out))
    torch.cuda.current_stream().wait_stream(side)
    return [out] + [t.grad for t in ts]


def _offloaded(fn, ts, dev):
    """Everything a step keeps goes to host memory and comes back."""
    with torch.autograd.graph.saved_tensors_hooks(lambda t: t.detach().cpu(), lambda t: t.to(dev)):
        out = fn(*ts)
    out.backward(_out_grad(out))
    return [out] + [t.grad for t in ts]


def _retained(fn, ts, dev):
    out = fn(*ts)
    out.backward(_out_grad(out), retain_graph=True)
    out.backward(_out_grad(out, seed=10))
    with pytest.raises(RuntimeError, match="second time"):
        out.backward(_out_grad(out))
    return [out] + [t.grad for t in ts]


def _strided(fn, ts, dev):
    ts = [t.detach().transpose(0, -1).contiguous().transpose(0, -1).requires_grad_(True) for t in ts]
    out = fn(*ts)
    out.backward(_out_grad(out)[:1, :1].expand_as(out))
    return [out] + [t.grad for t in ts]


def _one_leaf(fn, ts, dev):
    leaf = len(ts) - 2                                # (the weight)
    ts = [t.detach().requires_grad_(i == leaf) for i, t in enumerate(ts)]
    out = fn(*ts)
    out.backward(_out_grad(out))
    assert all(t.grad is None for i, t in enumerate(ts) if i != leaf)
    return [out, ts[leaf].grad]


class _NoGradient(torch.autograd.Function):
    @staticmethod
    def forward(ctx, x):
        return x.clone()

    @staticmethod
    def backward(ctx, g):
        return None


def _undefined(fn, ts, dev):
    """A consumer whose backward pass hands nothing on: gradients of zero, as for any Python autograd function."""
    out = fn(*ts)
    _NoGradient.apply(out).sum().backward()
    return [out] + [t.grad for t in ts]


SCENARIOS = {f.__name__.strip("_"): f for f in (_plain_step, _side_stream, _offloaded, _retained, _strided, _one_leaf, _undefined)}


@pytest.mark.parametrize("scenario", list(SCENARIOS))
@pytest.mark.parametrize("name", list(ENTRIES))
def test_native_and_python_routes_agree(name, scenario, dev, python_route):
    fn, tensors = ENTRIES[name]
    native = SCENARIOS[scenario](fn, _on(dev, tensors(4), True), dev)
    with python_route():
        python = SCENARIOS[scenario](fn, _on(dev, tensors(4), True), dev)
    if scenario != "strided":                         # (the route that was meant: non-contiguous tensors are Python's)
        assert native[0].grad_fn.name() != python[0].grad_fn.name() and "Function" not in native[0].grad_fn.name()
    tol = 4e-3 if python[0].dtype == torch.bfloat16 else 1e-5         # (atomics: sums in another order, one rounding)
    for i, (a, e) in enumerate(zip(native, python)):
        assert a is not None and e is not None, i
        assert a.dtype == e.dtype and a.shape == e.shape
        if scenario == "undefined" and i > 0:
            assert not a.any() and not e.any(), i
        else:
            assert rel_l2(a, e) < tol, (i, rel_l2(a, e))


@pytest.mark.parametrize("name", [n for n in ENTRIES if n != "depthwise"])
def test_differentiating_twice_is_an_error_on_both_routes(name, dev, python_route):
    fn, tensors = ENTRIES[name]
    def twice():
        ts = _on(dev, tensors(5), True)
        out = fn(*ts)
        gx = torch.autograd.grad(out, ts, _out_grad(out), create_graph=True)
        assert not any(g.requires_grad for g in gx)
        out = fn(*ts)
        for g in torch.autograd.grad(out, ts, _out_grad(out).requires_grad_(True), create_graph=True):
            with pytest.raises(RuntimeError, match="differentiate twice"):
                g.sum().backward(retain_graph=True)
    twice()
    with python_route():
        twice()


def test_what_native_code_leaves_to_python(dev, python_route):
    """Types to unify, arguments of other types: the same results, not an error."""
    fn, tensors = ENTRIES["conv3d_bf16"]
    x, off, m, w, b = _on(dev, tensors(6))
    want = fn(x, off, m, w, b)
    for args in ((x, off, m.double(), w.float(), b), (x, off, m, w, b.float())):
        assert rel_l2(fn(*args), want) < 4e-3
    assert rel_l2(_ops.deform_conv3d(x, off, m, w, b, 1.0, 1, 1, 1, 1, 1, 1, 1, 1, 1, 1), want) < 4e-3
    with pytest.raises(RuntimeError, match="ndimension"):
        fn(x, off, m, w, b[None])
    with pytest.raises(RuntimeError, match="offset.size"):
        fn(x, off[:, :3], m, w, b)


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
