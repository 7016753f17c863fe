"""Functional API and base modules, mirroring
ops/dconv-native/src/dconv_native/deform_conv.py of the reference: same names,
argument orders, parameter shapes and initialisation.
"""
import math

import torch
from torch import nn
from torch.nn import init
from torch.nn.modules.utils import _single, _triple
from torch.nn.parameter import Parameter

from . import _ops


def _any_half_inputs(*inputs):
    # deform_conv.py:15-16
    return any(t is not None and t.dtype == torch.half for t in inputs)


def _upcast_half(input, offset, alpha, weight, bias):
    # deform_conv.py:23-28 / :54-59: one float16 tensor makes the whole call float32
    if _any_half_inputs(input, offset, alpha, weight, bias):
        input = input.float()
        offset = offset.float()
        alpha = alpha.float() if alpha is not None else None
        weight = weight.float()
        bias = bias.float() if bias is not None else None
    return input, offset, alpha, weight, bias


def _float32_for_unchunked_bfloat16(input, offset, alpha, weight, bias, stride, padding, dilation, groups,
                                    offset_groups, offset_axes):
    """bfloat16 problems whose channel counts the bfloat16 matrix-core kernels cannot chunk (64 channels per weight
    group and per offset group: e.g. 256 channels in 8 offset groups) but the float32 ones can (32): the tensors as
    float32, and True -- the caller rounds the result back.  The direct kernels that would serve such a problem
    in bfloat16 are two to three orders of magnitude slower (N=2, C=256, 8 offset groups, 8x30x54: 493 + 695 ms
    against 0.7 + 2.0 ms).  Not in the reference."""
    if not (input.is_cuda and input.dtype == torch.bfloat16):
        return input, offset, alpha, weight, bias, False
    args = (input, offset, alpha, weight, stride, padding, dilation, groups, offset_groups, offset_axes)
    if _ops.conv3d_algo(*args) != "generic" or _ops.conv3d_algo(*args, as_dtype=torch.float32) != "mfma":
        return input, offset, alpha, weight, bias, False
    return (input.float(), offset.float(), alpha.float() if alpha is not None else None, weight.float(),
            bias.float() if bias is not None else None, True)


def _zero_channels_for_the_chunking(input, offset, alpha, weight, stride, padding, dilation, groups, offset_groups,
                                    offset_axes):
    """One weight group and one offset group whose channel count is no multiple of the matrix-core kernels' chunk (64
    bfloat16 / 32 float32 channels): input and weight padded with zero channels up to the next multiple, which changes
    no result (autograd drops the padding's gradient) and keeps the problem off the direct kernels.  Not in the
    reference."""
    if not input.is_cuda or groups != 1 or offset_groups != 1 or input.dtype not in (torch.bfloat16, torch.float32):
        return input, weight
    chunk = 64 if input.dtype == torch.bfloat16 else 32
    cin = input.shape[1]
    # (at least half a chunk of real channels: below that the direct kernels are not slow, and they are exact in
    # float32, which the tiny cases of the reference's own tests rely on)
    if cin % chunk == 0 or cin % chunk < chunk // 2 or _ops.conv3d_algo(input, offset, alpha, weight, stride, padding, dilation, 1, 1,
                                             offset_axes) != "generic":
        return input, weight
    extra = chunk - cin % chunk
    xp = torch.nn.functional.pad(input, (0, 0, 0, 0, 0, 0, 0, extra))
    wp = torch.nn.functional.pad(weight, (0, 0, 0, 0, 0, 0, 0, extra))
    if _ops.conv3d_algo(xp, offset, alpha, wp, stride, padding, dilation, 1, 1, offset_axes) != "mfma":
        return input, weight
    return xp, wp


def deform_conv1d(input, offset, alpha, weight, bias=None, stride=1, padding=0, dilation=1,
                  n_weight_groups=1, n_offset_groups=1):
    """deform_conv.py:19-40.  `alpha=None` means no modulation and `bias=None`
    no bias (the reference materialises ones / zeros for them, :30-35)."""
    if _any_half_inputs(input, offset, alpha, weight, bias):
        input, offset, alpha, weight, bias = _upcast_half(input, offset, alpha, weight, bias)
    return _ops.deform_conv1d(input, offset, alpha, weight, bias, stride, padding, dilation,
                              n_weight_groups, n_offset_groups)


def deform_conv3d(input, offset, alpha, weight, bias=None, stride=(1, 1, 1), padding=(0, 0, 0),
                  dilation=(1, 1, 1), n_weight_groups=1, n_offset_groups=1, output_relu=None, output_stats=False,
                  offset_axes=7, backward_memory="default", backward_slices=0, prepared=None, backward_f32_split=False):
    """deform_conv.py:42-85.  `output_relu` (not in the reference): None, or the scale s of an activation
    s * relu(.) that is applied to the output inside the forward kernels (1.0 for nn.ReLU, 1.71285855 for the
    ScaledReLU of network/layers.py:409-419).  `output_stats` (not in the reference): also return the float32
    [N, Cout, 2] sums and sums of squares of the output per (sample, channel), by a pass over it -- what the GroupNorm behind the convolution needs (network/modules/refinement.py:38-43).
    `offset_axes` (not in the reference): mask of the axes (1 z, 2 y, 4 x) along which the offsets displace; the
    other offset channels are read as zero and get zero gradient, which is what the Spatial / Temporal layers do to a
    copy of the tensor (dconv_native/modules.py:87-120).  Matrix-core kernels only.
    `backward_memory`, `backward_slices` (not in the reference; matrix-core kernels): how the
    backward pass trades workspace for time -- "default" (sampled columns in a buffer of their own: fastest),
    "in_place" (bfloat16: the columns written over the grad-column rows: about a third less workspace, a few per cent
    slower), "resample" (no columns: the grad-weight kernel samples again); `backward_slices` n >= 2 (bfloat16) runs
    the pass in n slices over the offset groups with buffers for one slice (least memory, slowest).  `prepared`: the calling
    layer's _ops.PreparedRegion (DeformConv3d.reuse_prepared), or None.  `backward_f32_split` (float32 problems on the
    matrix-core kernels): also the backward matrix kernels that by default stay on the float32 instruction (the
    grad-weight kernel that samples again, the 1-D operator's, the fallback data kernel) carry their float operands as
    two bfloat16 halves like the forward kernels do -- faster, gradients with a relative error of about 4e-6 of their
    scale instead of 1e-7.  The default grad-weight path (a product over sampled columns) is not affected."""
    from . import _lib
    flags = {"default": _lib.BWD_GW_DEFAULT, "columns": _lib.BWD_GW_COLUMNS, "in_place": _lib.BWD_GW_IN_PLACE,
             "resample": _lib.BWD_GW_RESAMPLE}[backward_memory] | _lib.bwd_slices(backward_slices)
    if backward_f32_split:
        flags |= _lib.BWD_F32_SPLIT
    if not output_relu and not output_stats and prepared is None:
        # (what the rest of this function prepares is for other calls than those that the native code takes)
        out = _ops._try_native("conv3d", input, offset, alpha, weight, bias, _triple(stride), _triple(padding), _triple(dilation),
                               n_weight_groups, n_offset_groups, offset_axes, flags, _ops._keep_max())
        if out is not None:
            return out
    input, offset, alpha, weight, bias = _upcast_half(input, offset, alpha, weight, bias)
    stride_d, stride_h, stride_w = _triple(stride)
    pad_d, pad_h, pad_w = _triple(padding)
    dilation_d, dilation_h, dilation_w = _triple(dilation)
    # shapes the matrix-core kernels do not chunk as they are: zero channels where that does it (one group), float32
    # for bfloat16 problems where that does
    input, weight = _zero_channels_for_the_chunking(
        input, offset, alpha, weight, (stride_d, stride_h, stride_w), (pad_d, pad_h, pad_w),
        (dilation_d, dilation_h, dilation_w), n_weight_groups, n_offset_groups, offset_axes)
    input, offset, alpha, weight, bias, rounded = _float32_for_unchunked_bfloat16(
        input, offset, alpha, weight, bias, (stride_d, stride_h, stride_w), (pad_d, pad_h, pad_w),
        (dilation_d, dilation_h, dilation_w), n_weight_groups, n_offset_groups, offset_axes)
    res = _ops.deform_conv3d(input, offset, alpha, weight, bias, stride_d, stride_h, stride_w,
                             pad_d, pad_h, pad_w, dilation_d, dilation_h, dilation_w,
                             n_weight_groups, n_offset_groups, float(output_relu) if output_relu else 0.0,
                             output_stats, offset_axes, flags, None if rounded else prepared)
    if rounded:     # (the statistics, float32 anyway, are those of the unrounded output)
        return (res[0].bfloat16(), res[1]) if output_stats else res.bfloat16()
    return res


def deform_conv3d_sized(input, size_map, alpha, weight, bias=None, mode="xyz", size_activation="linear",
                        stride=(1, 1, 1), padding=(0, 0, 0), dilation=(1, 1, 1), n_weight_groups=1, output_relu=None,
                        output_stats=False):
    """The deformable convolution of the size-conditioned layers (network/layers.py:184-313) as ONE operator:
    equal to deform_conv3d(input, offsets_from_size_map(size_activation(size_map), mode, kernel, dilation), alpha, ...)
    with one offset group, but the tap offsets are formed inside the sampler from the raw size prediction
    `size_map` [N, 3|2|2|1, Do, Ho, Wo] (mode "xyz" | "xxz" | "xy" | "x"); its gradient comes back in that shape.
    Half inputs are up-cast like in deform_conv3d."""
    if input.is_cuda and input.dtype != torch.half and not output_relu and not output_stats and mode.lower() in _ops._SIZE_CHANNELS:
        triples = tuple(_triple(t) for t in (stride, padding, dilation))
        out = _ops._try_native("conv3d_sized", input, size_map, alpha, weight, bias,
                               _ops._size_template(mode.lower(), tuple(weight.shape[2:]), triples[2], size_activation),
                               _ops._SIZE_CHANNELS[mode.lower()], *triples, n_weight_groups, _ops._keep_max())
        if out is not None:
            return out
    input, size_map, alpha, weight, bias = _upcast_half(input, size_map, alpha, weight, bias)
    # (the size map has the spatial shape of the offsets it stands for, which is all the question needs of it)
    input, size_map, alpha, weight, bias, rounded = _float32_for_unchunked_bfloat16(
        input, size_map, alpha, weight, bias, _triple(stride), _triple(padding), _triple(dilation), n_weight_groups, 1, 7)
    res = _ops.deform_conv3d_sized(input, size_map, alpha, weight, bias, mode, size_activation, stride, padding,
                                   dilation, n_weight_groups, float(output_relu) if output_relu else 0.0, output_stats)
    if rounded:
        return (res[0].bfloat16(), res[1]) if output_stats else res.bfloat16()
    return res


class DeformConvNd(nn.Module):
    """deform_conv.py:88-151."""

    def __init__(self, in_channels, out_channels, kernel_size, stride, padding, dilation, groups,
                 offset_groups, bias):
        super().__init__()
        if in_channels % groups != 0:
            raise ValueError("in_channels must be divisible by groups")
        if in_channels % offset_groups != 0:
            raise ValueError("in_channels must be divisible by offset_groups")
        if out_channels % groups != 0:
            raise ValueError("out_channels must be divisible by groups")
        self.in_channels = in_channels
        self.out_channels = out_channels
        self.kernel_size = kernel_size
        self.stride = stride
        self.padding = padding
        self.dilation = dilation
        self.groups = groups
        self.offset_groups = offset_groups
        self.weight = Parameter(torch.empty(out_channels, in_channels // groups, *kernel_size),
                                requires_grad=True)
        if bias:
            self.bias = Parameter(torch.empty(out_channels), requires_grad=True)
        else:
            self.register_parameter("bias", None)
        self.reset_parameters()

    def reset_parameters(self):
        # deform_conv.py:127-132, the initialisation of nn.Conv3d
        init.kaiming_uniform_(self.weight, a=math.sqrt(5))
        if self.bias is not None:
            fan_in, _ = init._calculate_fan_in_and_fan_out(self.weight)
            bound = 1 / math.sqrt(fan_in)
            init.uniform_(self.bias, -bound, bound)

    def extra_repr(self):
        s = f"{self.in_channels}, {self.out_channels}, kernel_size={self.kernel_size}, stride={self.stride}"
        if self.padding != (0,) * len(self.padding):
            s += f", padding={self.padding}"
        if self.dilation != (1,) * len(self.dilation):
            s += f", dilation={self.dilation}"
        if self.groups != 1:
            s += f", groups={self.groups}"
        if self.offset_groups != 1:
            s += f", offset_groups={self.offset_groups}"
        if self.bias is None:
            s += ", bias=False"
        return s


class DeformConv1d(DeformConvNd):
    """deform_conv.py:154-172."""

    def __init__(self, in_channels, out_channels, kernel_size, stride=1, padding=0, dilation=1,
                 groups=1, offset_groups=1, bias=True):
        super().__init__(in_channels, out_channels, _single(kernel_size), _single(stride),
                         _single(padding), _single(dilation), groups, offset_groups, bias)

    def forward(self, input, offset, alpha=None):
        return deform_conv1d(input, offset, alpha, self.weight, self.bias, self.stride[0],
                             self.padding[0], self.dilation[0], self.groups, self.offset_groups)


class DeformConv3d(DeformConvNd):
    """deform_conv.py:175-209.  `output_relu_scale` (None by default; set by util.fuse_output_activation) is
    the scale of a ReLU that the forward kernels apply to the output themselves."""
    output_relu_scale = None
    # set by util.fuse_conv_act_norm: the forward pass also keeps the per-channel sums of its output in
    # `last_output_stats` (float32 [N, Cout, 2]) for the GroupNorm behind it
    keep_output_stats = False
    last_output_stats = None
    # how the backward pass trades workspace for time (see deform_conv3d); plain attributes, settable per layer
    backward_memory = "default"
    backward_slices = 0
    # True: the layer keeps a device buffer (d2c_conv3d_prepared_bytes: the input's channels-last copy and the weights
    # in the matrix-core kernels' operand orders) between calls, so that the backward call of a step does not lay the
    # input out again and forward calls with unchanged weights (inference) do not re-order them.  Costs that buffer
    # (input-sized + twice the weights) per layer for as long as the layer lives.
    reuse_prepared = False
    _prepared = None
    backward_f32_split = False

    def __init__(self, in_channels, out_channels, kernel_size, stride=1, padding=0, dilation=1,
                 groups=1, offset_groups=1, bias=True):
        super().__init__(in_channels, out_channels, _triple(kernel_size), _triple(stride),
                         _triple(padding), _triple(dilation), groups, offset_groups, bias)

    def forward(self, input, offset, alpha=None, offset_axes=7):
        prepared = None
        if self.reuse_prepared:
            if self._prepared is None:
                from ._ops import PreparedRegion
                self._prepared = PreparedRegion()
            prepared = self._prepared
        out = deform_conv3d(input, offset, alpha, self.weight, self.bias, self.stride, self.padding,
                            self.dilation, self.groups, self.offset_groups, output_relu=self.output_relu_scale,
                            output_stats=self.keep_output_stats, offset_axes=offset_axes,
                            backward_memory=self.backward_memory, backward_slices=self.backward_slices,
                            prepared=prepared, backward_f32_split=self.backward_f32_split)
        if self.keep_output_stats:
            out, self.last_output_stats = out
        return out
