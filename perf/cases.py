"""What is timed of this package: calls of its public operators and layers as a network makes them, from a feature map
of a few hundred positions to a long clip, forward only (inference) and forward + backward (a training step's share of
one layer), in float32 and bfloat16.

A case is a dict of plain values:

  kind      "conv3d"      deform_conv3d (groups = cin: the channel-separated form)
            "sized"       deform_conv3d_sized, dynamic dilation: a size map per location and axis in place of offsets
            "conv1d"      deform_conv1d (the length in `w`)
            "depthwise"   depthwise_separable_conv3d, the plain channel-separated convolution of the backbone
            "layer"       MDConv3d: predicts its offsets and modulation itself
            "sized_layer" XYZSizeConditionedMDConv3d: predicts its size map and modulation itself
            "block"       Sequential(MDConv3d, ReLU, GroupNorm) of a decoder, after util.fuse_conv_act_norm
  n, cin, cout, t, h, w, kt, kh, kw, stride, dilation, groups, offset_groups   padding keeps the size at stride 1
  dtype     "f32" | "bf16"
  backward  all gradients too, of the input, the deformation and the parameters
  spread    standard deviation of the offsets in voxels ("sized": the largest dilation)
"""
import math

import torch

import d2conv3d_amd as d2c
from d2conv3d_amd.depthwise_conv import depthwise_separable_conv3d
from d2conv3d_amd.util import fuse_conv_act_norm

DTYPES = {"f32": torch.float32, "bf16": torch.bfloat16}


def _case(kind, n, cin, cout, t, h, w, kernel=(3, 3, 3), dtype="f32", backward=True, spread=1.5, stride=1, dilation=1,
          groups=1, offset_groups=1):
    kt, kh, kw = kernel
    return dict(kind=kind, n=n, cin=cin, cout=cout, t=t, h=h, w=w, kt=kt, kh=kh, kw=kw, stride=stride,
                dilation=dilation, groups=groups, offset_groups=offset_groups, dtype=dtype, backward=backward,
                spread=spread)


def listed():
    cases = {
        # inference on one small feature map: a call whose launches and host work count
        "conv3d small f32 infer": _case("conv3d", 1, 64, 64, 4, 14, 25, backward=False),
        # the first configuration of the benchmark: forward only, float32
        "conv3d c1 f32 infer": _case("conv3d", 1, 64, 64, 8, 32, 32, backward=False, spread=1.0),
        # temporal deformable convolution, a training step
        "conv1d f32 train": _case("conv1d", 4, 512, 512, 1, 1, 64, kernel=(1, 1, 3)),
        # the stage-32 map of a channel-separated backbone with deformable filters
        "conv3d depthwise f32 train": _case("conv3d", 2, 1024, 1024, 8, 15, 27, groups=1024),
        # the backbone's ordinary channel-separated convolution
        "depthwise f32 train": _case("depthwise", 2, 256, 256, 8, 56, 56, groups=256),
        # dynamic dilation, both precisions
        "sized bf16 train": _case("sized", 2, 256, 256, 8, 30, 54, dtype="bf16", spread=4.0),
        "sized f32 train": _case("sized", 2, 256, 256, 8, 30, 54, spread=4.0),
        # modulated deformable convolution with eight offset groups, the headline
        "conv3d c3 bf16 train": _case("conv3d", 2, 512, 512, 8, 30, 54, dtype="bf16", spread=2.0, offset_groups=8),
        # a decoder's refinement layer behind a 1024-channel stage, with its own deformation branch
        "sized layer bf16 train": _case("sized_layer", 1, 1024, 256, 8, 30, 54, dtype="bf16", spread=1.0),
        # one arm of the decoder's global-convolution bridge
        "bridge bf16 train": _case("conv3d", 1, 2048, 256, 8, 30, 54, kernel=(1, 7, 1), dtype="bf16"),
        # a decoder block at stride 8 in inference, an odd width
        "block bf16 infer": _case("block", 1, 256, 256, 8, 60, 107, dtype="bf16", backward=False, spread=1.0),
        # a long clip
        "conv3d long clip bf16 train": _case("conv3d", 1, 256, 256, 32, 60, 108, dtype="bf16", spread=1.0),
    }
    return [dict(case, name=name) for name, case in cases.items()]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, round(math.exp(rng.uniform(math.log(lo), math.log(hi))))))


def draw(rng):
    most = max(_weight(c) for c in listed())
    most_bytes = max(work(c)["bytes"] for c in listed())
    while True:
        kind = rng.choice(["conv3d", "conv3d", "conv3d", "sized", "sized", "conv1d", "depthwise", "layer",
                           "sized_layer", "block"])
        dtype = rng.choice(["f32", "bf16"])
        backward = rng.random() < 0.6
        n = rng.choice([1, 1, 1, 2, 2, 3, 4])
        t, h = _log_int(rng, 2, 32), _log_int(rng, 7, 120)
        w = max(7, round(h * rng.uniform(0.9, 1.9)))
        cin, cout = (rng.choice([64, 64, 128, 192, 256, 256, 320, 512, 1024, 2048]),
                     rng.choice([64, 128, 192, 256, 256, 512]))
        kernel, stride, dilation, groups, offset_groups = (3, 3, 3), 1, 1, 1, 1
        spread = round(rng.uniform(0.5, 2.5), 2)
        if kind == "conv1d":
            t, h, w, kernel = 1, 1, _log_int(rng, 16, 1500), (1, 1, rng.choice([3, 3, 5]))
            dtype = "f32" if rng.random() < 0.7 else "bf16"
        elif kind == "depthwise":
            cin = cout = groups = rng.choice([64, 128, 256, 512, 1024])
            stride = rng.choice([1, 1, 1, 2])
        elif kind == "conv3d":
            form = rng.choice(["plain", "plain", "groups", "bridge", "separated", "dilated"])
            if form == "groups":
                offset_groups = rng.choice([g for g in (2, 4, 8) if cin % (64 * g) == 0] or [1])
            elif form == "bridge":
                kernel = rng.choice([(1, 7, 1), (1, 1, 7)])
            elif form == "separated":
                cin = cout = groups = rng.choice([64, 256, 512, 1024])
                dtype = "f32"
            elif form == "dilated":
                stride, dilation = rng.choice([(1, 2), (2, 1)])
        elif kind == "sized":
            spread = round(rng.uniform(2.0, 4.0), 2)
        elif kind == "layer":
            offset_groups = rng.choice([1, 1] + [g for g in (4, 8) if cin % (64 * g) == 0])
        if kind in ("layer", "sized_layer", "block"):
            # (mixed-precision networks; in float32 a layer's own branch is the stock convolution)
            dtype, spread = "bf16", 1.0
        case = _case(kind, n, cin, cout, t, h, w, kernel, dtype, backward, spread, stride, dilation, groups,
                     offset_groups)
        if _weight(case) <= most and work(case)["bytes"] <= most_bytes:
            return case


def _dims(c):
    """Output extents (the padding keeps the size at stride 1)."""
    return [(d - 1) // c["stride"] + 1 for d in (c["t"], c["h"], c["w"])]


def _taps(c):
    return c["kt"] * c["kh"] * c["kw"]


def _branch_channels(c):
    """Channels that a layer's own convolution predicts."""
    if c["kind"] == "sized_layer":
        return 3 + _taps(c)
    return 4 * c["offset_groups"] * _taps(c) if c["kind"] in ("layer", "block") else 0


def _flops(c):
    do, ho, wo = _dims(c)
    per_output = 2.0 * c["n"] * do * ho * wo * (c["cin"] // c["groups"]) * _taps(c)
    return per_output * (c["cout"] + _branch_channels(c)) * (3 if c["backward"] else 1)


def _weight(c):
    """How much a case costs, roughly: its multiplications (a float32 one counts like four), and what the sampled
    values of a channel-separated form cost beside its few multiplications."""
    flops = _flops(c) * (4 if c["dtype"] == "f32" else 1)
    if c["kind"] == "conv3d" and c["groups"] > 1:
        flops *= 150
    do, ho, wo = _dims(c)
    sampled = 300.0 * c["n"] * do * ho * wo * c["cin"] * _taps(c) if c["kind"] not in ("depthwise", "conv1d") else 0.0
    return flops + sampled


def _elements(c):
    """Element counts of the tensors of a case: input, deformation inputs, output, parameters."""
    do, ho, wo = _dims(c)
    positions = c["n"] * do * ho * wo
    k, g = _taps(c), c["offset_groups"]
    x = c["n"] * c["cin"] * c["t"] * c["h"] * c["w"]
    axes = 1 if c["kind"] == "conv1d" else 3
    deformation = {"conv3d": (axes + 1) * g * k, "conv1d": (axes + 1) * g * k, "sized": 3 + k}.get(c["kind"], 0)
    params = c["cout"] * (c["cin"] // c["groups"]) * k + c["cout"]
    params += _branch_channels(c) * (c["cin"] * k + 1) + (2 * c["cout"] if c["kind"] == "block" else 0)
    return x, positions * deformation, positions * c["cout"], params


def work(case):
    x, deformation, out, params = _elements(case)
    size = 2 if case["dtype"] == "bf16" else 4
    count = x + deformation + params + out
    if case["backward"]:
        # grad_out and the inputs again (backward runs later, in a network), a gradient for each
        count += out + 2 * (x + deformation + params)
    return {"bytes": float(count * size), "flops": _flops(case)}


def tolerance(case):
    if case["dtype"] == "f32":
        return {"rel": 1e-5}
    # (the offsets that a layer predicts are rounded to bfloat16: with another order of its sums a sampling point now
    # and then lies on the other side of a voxel's boundary, where the offset's gradient jumps)
    return {"rel": 2e-2 if case["backward"] and _branch_channels(case) else 1e-2}


def prepare(case, seed):
    c, dev, dtype = case, torch.device("cuda"), DTYPES[case["dtype"]]
    gen = torch.Generator(device=dev).manual_seed(int(seed))
    grad = c["backward"]

    def normal(*shape, std=1.0):
        return (torch.randn(*shape, generator=gen, device=dev) * std).to(dtype)

    def uniform(*shape, lo, hi):
        return (torch.rand(*shape, generator=gen, device=dev) * (hi - lo) + lo).to(dtype)

    n, cin, cout, k, g = c["n"], c["cin"], c["cout"], _taps(c), c["offset_groups"]
    kernel = (c["kt"], c["kh"], c["kw"])
    padding = tuple(c["dilation"] * (v // 2) for v in kernel)
    bound = 1.0 / math.sqrt(cin // c["groups"] * k)
    dims, out_dims = (c["t"], c["h"], c["w"]), _dims(c)
    state = {"case": c}
    if c["kind"] == "conv1d":
        kernel, padding, dims, out_dims = kernel[2:], padding[2:], dims[2:], out_dims[2:]
    state["geometry"] = (c["stride"], padding, c["dilation"])
    x = normal(n, cin, *dims)
    if c["kind"] in ("layer", "sized_layer", "block"):
        cls = d2c.XYZSizeConditionedMDConv3d if c["kind"] == "sized_layer" else d2c.MDConv3d
        layer = cls(cin, cout, kernel, c["stride"], padding, c["dilation"], c["groups"], g)
        module = layer
        if c["kind"] == "block":
            module = torch.nn.Sequential(layer, torch.nn.ReLU(), torch.nn.GroupNorm(32, cout))
        module = module.to(dev, dtype)
        with torch.no_grad():
            layer.deform_conv.weight.copy_(uniform(*layer.deform_conv.weight.shape, lo=-bound, hi=bound))
            layer.deform_conv.bias.copy_(uniform(cout, lo=-bound, hi=bound))
            # a branch as training leaves it: deformations of about a voxel
            layer.deform_params.weight.copy_(normal(*layer.deform_params.weight.shape, std=c["spread"] * bound))
            if c["kind"] == "block":
                module[2].weight.copy_(uniform(cout, lo=0.5, hi=1.5))
                module[2].bias.copy_(uniform(cout, lo=-0.5, hi=0.5))
        if c["kind"] == "block":
            holder = torch.nn.ModuleList([module])
            fuse_conv_act_norm(holder)
            module = holder[0]
        inputs = [x]
        state["module"] = module.train(grad)
        state["params"] = [p for p in module.parameters()]
    else:
        weight = uniform(cout, cin // c["groups"], *kernel, lo=-bound, hi=bound)
        bias = uniform(cout, lo=-bound, hi=bound)
        if c["kind"] == "depthwise":
            inputs = [x, weight, bias]
        else:
            axes = 1 if c["kind"] == "conv1d" else 3
            if c["kind"] == "sized":
                deformation = uniform(n, 3, *out_dims, lo=0.5, hi=c["spread"])
            else:
                deformation = normal(n, axes * g * k, *out_dims, std=c["spread"])
            mask = torch.sigmoid(normal(n, g * k, *out_dims))
            inputs = [x, deformation, mask, weight, bias]
        state["params"] = []
    state["inputs"] = [v.requires_grad_(grad) for v in inputs]
    if grad:
        state["grad_out"] = normal(n, cout, *out_dims)
    return state


def _forward(state):
    c, inputs = state["case"], state["inputs"]
    stride, padding, dilation = state["geometry"]
    if "module" in state:
        return state["module"](*inputs)
    if c["kind"] == "conv3d":
        return d2c.deform_conv3d(*inputs, stride, padding, dilation, c["groups"], c["offset_groups"])
    if c["kind"] == "conv1d":
        return d2c.deform_conv1d(*inputs, stride, padding, dilation, c["groups"], c["offset_groups"])
    if c["kind"] == "sized":
        return d2c.deform_conv3d_sized(*inputs, mode="xyz", stride=stride, padding=padding, dilation=dilation)
    return depthwise_separable_conv3d(*inputs, stride, padding, dilation)


def run(state):
    if not state["case"]["backward"]:
        with torch.no_grad():
            return _forward(state)
    out = _forward(state)
    return (out.detach(),) + torch.autograd.grad(out, state["inputs"] + state["params"], state["grad_out"])
