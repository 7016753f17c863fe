// The operators' calls and their autograd nodes in native code: what d2conv3d_amd/_ops.py and depthwise_conv.py do in Python
// for every argument, for the calls that need nothing special.  A function here returns None for a call it does not
// take -- an argument that fails a check, tensors of types to be unified, non-contiguous or wrapped tensors, calls
// without a kernel of their own -- and the Python code then does it, with its conversions and its error messages.
//
// (Why: a forward call cost 55 us of host time and forward + backward 150 - 215 us, most of it interpreting Python, where
// the kernels of a small problem take 40 - 100 us.)
#include <Python.h>
#include <c10/core/DeviceGuard.h>
#include <c10/hip/HIPStream.h>
#include <hip/hip_runtime_api.h>
#include <torch/csrc/autograd/function.h>
#include <torch/csrc/autograd/functions/basic_ops.h>
#include <torch/csrc/autograd/functions/utils.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/autograd/saved_variable.h>
#include <torch/csrc/jit/frontend/tracer.h>
#include <torch/csrc/utils/pybind.h>
#include <torch/types.h>

#include <array>
#include <cstring>
#include <optional>

#include "../../../include/d2conv.h"

namespace py = pybind11;
using at::Tensor;
using torch::autograd::Node;
using torch::autograd::SavedVariable;
using torch::autograd::variable_list;
typedef std::array<int, 3> int3_t;
typedef std::optional<Tensor> opt_tensor;

namespace {

// _ops._WS_CACHE ((device index, stream) -> workspace tensor), the switch of that cache, and _ops._workspace
PyObject *g_ws_cache = nullptr, *g_ws_on = nullptr, *g_ws_make = nullptr;

void check(int rc, const char *what)
{
    if (rc != D2C_OK) throw std::runtime_error(std::string(what) + ": " + d2c_last_error() + " (code " + std::to_string(rc) + ")");
}
// (a tensor whose memory the kernels can take as it is: no subclass with its own dispatch, no functorch wrapper, no
// forward-mode tangent; and no call that torch.jit.trace records: of one it would see the allocation of the result
// alone, where the Python functions are recorded as operations)
bool plain(const Tensor &t)
{
    return t.defined() && !torch::jit::tracer::isTracing() && t.is_cuda() && t.layout() == at::kStrided && t.has_storage() && !t.unsafeGetTensorImpl()->is_python_dispatch() &&
           t.is_contiguous() && !t._fw_grad(0).defined();
}
int dtype_code(const Tensor &t)
{
    switch (t.scalar_type()) {
    case at::kFloat: return D2C_F32;
    case at::kDouble: return D2C_F64;
    case at::kBFloat16: return D2C_BF16;
    default: return -1;
    }
}
void *ptr(const Tensor &t) { return t.defined() ? t.data_ptr() : nullptr; }
void *ptr_at(const Tensor &t, int64_t channel)
{
    return t.defined() ? (char *)t.data_ptr() + channel * t.stride(1) * t.element_size() : nullptr;
}
hipStream_t stream_of(const Tensor &t) { return c10::hip::getCurrentHIPStream(t.device().index()).stream(); }

// The workspace of a call: the one kept for this device and stream where it is large enough
Tensor workspace(size_t bytes, const Tensor &like, hipStream_t st)
{
    if (bytes == 0) return Tensor();
    hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
    if (hipStreamIsCapturing(st, &cap) != hipSuccess || cap != hipStreamCaptureStatusNone)
        return at::empty({(int64_t)bytes}, like.options().dtype(at::kByte).requires_grad(false));
    py::gil_scoped_acquire gil;
    if (PyObject_IsTrue(PyList_GET_ITEM(g_ws_on, 0)) == 1) {
        py::tuple key = py::make_tuple((int)like.device().index(), (uintptr_t)st);
        PyObject *have = PyDict_GetItem(g_ws_cache, key.ptr());
        if (have && THPVariable_Check(have)) {
            const Tensor &ws = THPVariable_Unpack(have);
            if ((size_t)ws.numel() >= bytes) return ws;
        }
    }
    py::object made = py::reinterpret_steal<py::object>(PyObject_CallFunction(g_ws_make, "KN", (unsigned long long)bytes,
                                                                              THPDevice_New(like.device())));
    if (!made) throw py::error_already_set();
    return THPVariable_Unpack(made.ptr());
}

// ... of a forward call that keeps no columns.  What it takes beyond the least it runs with, to hold the columns in, is not
// kept from call to call, and a call that does not get it runs with the least.
Tensor forward_workspace(size_t &bytes, const d2c_conv3d_desc &q, const d2c_size_map_desc *sz, const Tensor &like, hipStream_t st)
{
    const size_t least = d2c_conv3d_forward_least_workspace_bytes(&q, sz);
    if (bytes > least) {
        try {
            return at::empty({(int64_t)bytes}, like.options().dtype(at::kByte).requires_grad(false));
        } catch (const c10::OutOfMemoryError &) {
            bytes = least;
        }
    }
    return workspace(bytes, like, st);
}

Tensor no_grad_empty_like(const Tensor &t) { return at::empty(t.sizes(), t.options().requires_grad(false)); }

// Gradients that leave a node while a graph of the backward pass is being recorded through its grad_out: differentiating
// them is an error (torch's once_differentiable).
void once_differentiable(variable_list &grads, const Tensor &grad_out)
{
    if (!at::GradMode::is_enabled() || !grad_out.requires_grad()) return;
    auto err = std::make_shared<torch::autograd::DelayedError>(
        "trying to differentiate twice a function that was marked with @once_differentiable", 1);
    for (auto &g : grads)
        if (g.defined()) {
            Tensor v = g.detach();
            v.requires_grad_(true);
            variable_list out = (*err)(variable_list{v});
            g = out[0];
        }
}

template <class NodeT> Tensor record(Tensor out, const std::shared_ptr<NodeT> &node)
{
    torch::autograd::set_history(out, node);
    return out;
}
template <class... T> bool wants_grad(const T &...t) { return at::GradMode::is_enabled() && torch::autograd::compute_requires_grad(t...); }

// ---------------------------------------------------------------- deform_conv3d, sized and packed
enum Form { OFFSETS, SIZED, PACKED };
struct Call3d {
    d2c_conv3d_desc desc;
    d2c_size_map_desc size;
    Form form;
    bool sized;
    int64_t lead;                    // PACKED: channels in front of the modulation values
    const d2c_size_map_desc *sz() const { return sized ? &size : nullptr; }
};

Tensor forward_3d(const Call3d &c, const Tensor &x, const Tensor &off, const Tensor &alpha, const Tensor &w, const Tensor &bias,
                  bool keep, size_t keep_max, Tensor &columns)
{
    const d2c_conv3d_desc &q = c.desc;
    check(d2c_conv3d_check(&q), c.form == OFFSETS ? "deform_conv3d" : (c.form == SIZED ? "deform_conv3d_sized" : "deform_conv3d_packed"));
    c10::DeviceGuard guard(x.device());
    const hipStream_t st = stream_of(x);
    Tensor out = at::empty({q.N, q.Cout, q.Do, q.Ho, q.Wo}, x.options().requires_grad(false));
    if (keep) {
        const size_t n = d2c_conv3d_keep_bytes(&q, c.sz());
        if (n > 0 && n <= keep_max) {
            try {
                columns = at::empty({(int64_t)n}, x.options().dtype(at::kByte).requires_grad(false));
            } catch (const c10::OutOfMemoryError &) {      // (no room to keep them: the backward pass samples again)
            }
        }
    }
    size_t nb = columns.defined() ? d2c_conv3d_forward_keep_workspace_bytes(&q, c.sz())
                : c.sized ? d2c_conv3d_sized_forward_workspace_bytes(&q, &c.size) : d2c_conv3d_forward_workspace_bytes(&q);
    const Tensor ws = columns.defined() ? workspace(nb, x, st) : forward_workspace(nb, q, c.sz(), x, st);
    const void *po = ptr(off), *pm = c.form == PACKED ? ptr_at(off, c.lead) : ptr(alpha);
    int rc;
    if (columns.defined())
        rc = d2c_conv3d_forward_columns(&q, c.sz(), ptr(x), po, pm, ptr(w), ptr(bias), ptr(out), ptr(columns), columns.numel(), ptr(ws), nb, st);
    else if (c.sized) rc = d2c_conv3d_sized_forward(&q, &c.size, ptr(x), po, pm, ptr(w), ptr(bias), ptr(out), ptr(ws), nb, st);
    else rc = d2c_conv3d_forward(&q, ptr(x), po, pm, ptr(w), ptr(bias), ptr(out), ptr(ws), nb, st);
    check(rc, c.form == OFFSETS ? "deform_conv3d forward" : (c.form == SIZED ? "deform_conv3d_sized forward" : "deform_conv3d_packed forward"));
    return out;
}

// inputs: x, offsets | size map | deformation, mask, weight, bias
struct DeformConv3dBackward : public Node {
    Call3d c;
    SavedVariable x, off, alpha, w, kept;
    bool has_alpha = false, has_bias = false, has_columns = false;
    std::string name() const override { return "DeformConv3dBackward"; }
    void release_variables() override
    {
        const std::lock_guard<std::mutex> lock(mutex_);
        x.reset_data(); off.reset_data(); alpha.reset_data(); w.reset_data(); kept.reset_data();
    }
    variable_list apply(variable_list &&grads) override
    {
        variable_list r(5);
        const std::lock_guard<std::mutex> lock(mutex_);
        if (!grads[0].defined()) grads[0] = input_metadata(0).zeros_like();
        {
            at::NoGradGuard no_grad;
            const Tensor vx = x.unpack(), vo = off.unpack(), va = has_alpha ? alpha.unpack() : Tensor(), vw = w.unpack();
            const Tensor columns = has_columns ? kept.unpack() : Tensor();
            c10::DeviceGuard guard(vx.device());
            const hipStream_t st = stream_of(vx);
            const Tensor g = grads[0].contiguous().to(vx.scalar_type());
            const d2c_conv3d_desc &q = c.desc;
            if (should_compute_output(0)) r[0] = no_grad_empty_like(vx);
            if (should_compute_output(1)) r[1] = no_grad_empty_like(vo);
            if (has_alpha && should_compute_output(2)) r[2] = no_grad_empty_like(va);
            if (should_compute_output(3)) r[3] = no_grad_empty_like(vw);
            if (has_bias && should_compute_output(4)) r[4] = at::empty({q.Cout}, vw.options().requires_grad(false));
            const void *pm = c.form == PACKED ? ptr_at(vo, c.lead) : ptr(va);
            void *gm = c.form == PACKED ? ptr_at(r[1], c.lead) : ptr(r[2]);
            const size_t nb = columns.defined() ? d2c_conv3d_backward_keep_workspace_bytes(&q, c.sz())
                              : c.sized ? d2c_conv3d_sized_backward_workspace_bytes(&q, &c.size) : d2c_conv3d_backward_workspace_bytes(&q);
            const Tensor ws = workspace(nb, vx, st);
            int rc;
            if (columns.defined())
                rc = d2c_conv3d_backward_columns(&q, c.sz(), ptr(g), ptr(vx), ptr(vo), pm, ptr(vw), ptr(columns), columns.numel(), ptr(r[0]),
                                                 ptr(r[1]), gm, ptr(r[3]), ptr(r[4]), ptr(ws), nb, st);
            else if (c.sized)
                rc = d2c_conv3d_sized_backward(&q, &c.size, ptr(g), ptr(vx), ptr(vo), pm, ptr(vw), ptr(r[0]), ptr(r[1]), gm, ptr(r[3]),
                                               ptr(r[4]), ptr(ws), nb, st);
            else
                rc = d2c_conv3d_backward(&q, ptr(g), ptr(vx), ptr(vo), pm, ptr(vw), ptr(r[0]), ptr(r[1]), gm, ptr(r[3]), ptr(r[4]), ptr(ws),
                                         nb, st);
            check(rc, c.form == OFFSETS ? "deform_conv3d backward" : (c.form == SIZED ? "deform_conv3d_sized backward" : "deform_conv3d_packed backward"));
        }
        once_differentiable(r, grads[0]);
        return r;
    }
};

// everything the Python checks ask for (_ops._check_common, _unify), or false
bool fill_3d(Call3d &c, const Tensor &x, const Tensor &off, const Tensor &alpha, const Tensor &w, const Tensor &bias, const int3_t &s,
             const int3_t &p, const int3_t &d, int64_t groups, int64_t G, int64_t axes, int64_t flags, int64_t mask_act)
{
    if (!plain(x) || !plain(off) || !plain(w) || (alpha.defined() && !plain(alpha)) || (bias.defined() && !plain(bias))) return false;
    if (x.dim() != 5 || off.dim() != 5 || w.dim() != 5 || (alpha.defined() && alpha.dim() != 5) || (bias.defined() && bias.dim() != 1)) return false;
    const at::Device dev = x.device();
    if (off.device() != dev || w.device() != dev || (alpha.defined() && alpha.device() != dev) || (bias.defined() && bias.device() != dev)) return false;
    const int dt = dtype_code(x), adt = dtype_code(off);
    if (dt < 0 || dtype_code(w) != dt || (bias.defined() && dtype_code(bias) != dt) || (alpha.defined() && dtype_code(alpha) != adt)) return false;
    if (adt != dt && !(dt == D2C_BF16 && adt == D2C_F32)) return false;
    if (groups < 1 || G < 1 || w.size(0) % groups || w.size(1) * groups != x.size(1) || w.size(0) % G || x.size(1) % G) return false;
    const int64_t K = w.size(2) * w.size(3) * w.size(4), lim = 1ll << 31;
    if (off.size(0) != x.size(0) || (bias.defined() && bias.size(0) != w.size(0))) return false;
    if (alpha.defined() && (alpha.size(0) != x.size(0) || alpha.size(1) != G * K || alpha.sizes().slice(2) != off.sizes().slice(2))) return false;
    if (c.form == OFFSETS && off.size(1) != 3 * G * K) return false;
    if (c.form == PACKED && off.size(1) != c.lead + G * K) return false;
    for (const Tensor *t : {&x, &off, &w})
        for (int64_t v : t->sizes())
            if (v < 1 || v >= lim) return false;
    d2c_conv3d_desc &q = c.desc;
    std::memset(&q, 0, sizeof q);
    q.N = (int)x.size(0); q.Cin = (int)x.size(1); q.Cout = (int)w.size(0);
    q.D = (int)x.size(2); q.H = (int)x.size(3); q.W = (int)x.size(4);
    q.kd = (int)w.size(2); q.kh = (int)w.size(3); q.kw = (int)w.size(4);
    q.sd = s[0]; q.sh = s[1]; q.sw = s[2]; q.pd = p[0]; q.ph = p[1]; q.pw = p[2]; q.dd = d[0]; q.dh = d[1]; q.dw = d[2];
    q.groups = (int)groups; q.offset_groups = (int)G;
    q.Do = (int)off.size(2); q.Ho = (int)off.size(3); q.Wo = (int)off.size(4);
    q.dtype = dt; q.aux_dtype = adt;
    q.epilogue = D2C_EPILOGUE_NONE; q.epilogue_scale = 1.f;
    q.offset_axes = (int)axes; q.backward_flags = (int)flags;
    if (c.form == PACKED) { q.deform_channels = (int)off.size(1); q.mask_activation = (int)mask_act; }
    return true;
}

py::object run_3d(Call3d &c, const Tensor &x, const Tensor &off, const Tensor &alpha, const Tensor &w, const Tensor &bias, int64_t keep_max)
{
    const bool grad = wants_grad(x, off, alpha, w, bias);
    Tensor columns;
    std::shared_ptr<DeformConv3dBackward> node;
    if (grad) {
        node = std::shared_ptr<DeformConv3dBackward>(new DeformConv3dBackward(), torch::autograd::deleteNode);
        node->set_next_edges(torch::autograd::collect_next_edges(x, off, alpha, w, bias));
    }
    Tensor out = forward_3d(c, x, off, alpha, w, bias, grad && w.requires_grad() && keep_max > 0, (size_t)keep_max, columns);
    if (!grad) return py::cast(out);
    node->c = c;
    node->x = SavedVariable(x, false); node->off = SavedVariable(off, false); node->w = SavedVariable(w, false);
    node->has_alpha = alpha.defined(); node->has_bias = bias.defined();
    if (alpha.defined()) node->alpha = SavedVariable(alpha, false);
    node->has_columns = columns.defined();
    if (columns.defined()) node->kept = SavedVariable(columns, false);
    return py::cast(record(out, node));
}

py::object conv3d(const Tensor &x, const Tensor &off, const opt_tensor &alpha, const Tensor &w, const opt_tensor &bias, int3_t s, int3_t p,
                  int3_t d, int64_t groups, int64_t G, int64_t axes, int64_t flags, int64_t keep_max)
{
    Call3d c;
    c.form = OFFSETS; c.sized = false; c.lead = 0;
    const Tensor a = alpha.value_or(Tensor()), b = bias.value_or(Tensor());
    if (!fill_3d(c, x, off, a, w, b, s, p, d, groups, G, axes, flags, 0)) return py::none();
    // (the direct kernels' problems: Python may pad or convert them to ones that the matrix-core kernels take)
    const int algo = d2c_conv3d_algo(&c.desc);
    if (algo != D2C_ALGO_MFMA && algo != D2C_ALGO_DEPTHWISE) return py::none();
    return run_3d(c, x, off, a, w, b, keep_max);
}
// `size`: the bytes of a d2c_size_map_desc whose N, P and dtype are filled in here
bool size_desc(Call3d &c, const std::string &size, const Tensor &map)
{
    if (size.size() != sizeof c.size) return false;
    std::memcpy(&c.size, size.data(), sizeof c.size);
    c.size.N = c.desc.N; c.size.P = c.desc.Do * c.desc.Ho * c.desc.Wo;
    c.size.dtype = dtype_code(map) == D2C_BF16 ? D2C_BF16 : D2C_F32;
    c.sized = true;
    return true;
}
py::object conv3d_sized(const Tensor &x, const Tensor &map, const opt_tensor &alpha, const Tensor &w, const opt_tensor &bias,
                        const std::string &size, int64_t channels, int3_t s, int3_t p, int3_t d, int64_t groups, int64_t keep_max)
{
    Call3d c;
    c.form = SIZED; c.lead = 0;
    const Tensor a = alpha.value_or(Tensor()), b = bias.value_or(Tensor());
    if (!fill_3d(c, x, map, a, w, b, s, p, d, groups, 1, 7, 0, 0) || map.size(1) != channels || !size_desc(c, size, map)) return py::none();
    // (offset_axes of the description: all, as in the Python call, which leaves the field zero)
    c.desc.offset_axes = 0;
    if (d2c_conv3d_algo(&c.desc) != D2C_ALGO_MFMA) return py::none();
    return run_3d(c, x, map, a, w, b, keep_max);
}
py::object conv3d_packed(const Tensor &x, const Tensor &deformation, const Tensor &w, const opt_tensor &bias, int64_t lead, int64_t mask_act,
                         const std::string &size, int3_t s, int3_t p, int3_t d, int64_t groups, int64_t G, int64_t axes, int64_t flags,
                         int64_t keep_max)
{
    Call3d c;
    c.form = PACKED; c.lead = lead; c.sized = false;
    const Tensor none, b = bias.value_or(Tensor());
    if (!fill_3d(c, x, deformation, none, w, b, s, p, d, groups, G, axes, flags, mask_act)) return py::none();
    if (!size.empty() && !size_desc(c, size, deformation)) return py::none();
    c10::DeviceGuard guard(x.device());
    if (!d2c_conv3d_packed_supported(&c.desc, c.sz())) return py::none();
    return run_3d(c, x, deformation, none, w, b, keep_max);
}

// ---------------------------------------------------------------- deform_conv1d
struct DeformConv1dBackward : public Node {
    d2c_conv1d_desc q;
    SavedVariable x, off, alpha, w;
    bool has_alpha = false, has_bias = false;
    std::string name() const override { return "DeformConv1dBackward"; }
    void release_variables() override
    {
        const std::lock_guard<std::mutex> lock(mutex_);
        x.reset_data(); off.reset_data(); alpha.reset_data(); w.reset_data();
    }
    variable_list apply(variable_list &&grads) override
    {
        variable_list r(5);
        const std::lock_guard<std::mutex> lock(mutex_);
        if (!grads[0].defined()) grads[0] = input_metadata(0).zeros_like();
        {
            at::NoGradGuard no_grad;
            const Tensor vx = x.unpack(), vo = off.unpack(), va = has_alpha ? alpha.unpack() : Tensor(), vw = w.unpack();
            c10::DeviceGuard guard(vx.device());
            const hipStream_t st = stream_of(vx);
            const Tensor g = grads[0].contiguous().to(vx.scalar_type());
            if (should_compute_output(0)) r[0] = no_grad_empty_like(vx);
            if (should_compute_output(1)) r[1] = no_grad_empty_like(vo);
            if (has_alpha && should_compute_output(2)) r[2] = no_grad_empty_like(va);
            if (should_compute_output(3)) r[3] = no_grad_empty_like(vw);
            if (has_bias && should_compute_output(4)) r[4] = at::empty({q.Cout}, vw.options().requires_grad(false));
            const size_t nb = d2c_conv1d_backward_workspace_bytes(&q);
            const Tensor ws = workspace(nb, vx, st);
            check(d2c_conv1d_backward(&q, ptr(g), ptr(vx), ptr(vo), ptr(va), ptr(vw), ptr(r[0]), ptr(r[1]), ptr(r[2]), ptr(r[3]), ptr(r[4]),
                                      ptr(ws), nb, st), "deform_conv1d backward");
        }
        once_differentiable(r, grads[0]);
        return r;
    }
};

py::object conv1d(const Tensor &x, const Tensor &off, const opt_tensor &alpha, const Tensor &w, const opt_tensor &bias, int64_t s, int64_t p,
                  int64_t d, int64_t groups, int64_t G, bool quirks)
{
    const Tensor a = alpha.value_or(Tensor()), b = bias.value_or(Tensor());
    if (!plain(x) || !plain(off) || !plain(w) || (a.defined() && !plain(a)) || (b.defined() && !plain(b))) return py::none();
    if (x.dim() != 3 || off.dim() != 3 || w.dim() != 3 || (a.defined() && a.dim() != 3) || (b.defined() && b.dim() != 1)) return py::none();
    const at::Device dev = x.device();
    if (off.device() != dev || w.device() != dev || (a.defined() && a.device() != dev) || (b.defined() && b.device() != dev)) return py::none();
    const int dt = dtype_code(x), adt = dtype_code(off);
    if (dt < 0 || dtype_code(w) != dt || (b.defined() && dtype_code(b) != dt) || (a.defined() && dtype_code(a) != adt)) return py::none();
    if (adt != dt && !(dt == D2C_BF16 && adt == D2C_F32)) return py::none();
    if (groups < 1 || G < 1 || w.size(0) % groups || w.size(1) * groups != x.size(1) || w.size(0) % G || x.size(1) % G) return py::none();
    const int64_t K = w.size(2), lim = 1ll << 31;
    if (off.size(0) != x.size(0) || off.size(1) != G * K || (b.defined() && b.size(0) != w.size(0))) return py::none();
    if (a.defined() && (a.size(0) != x.size(0) || a.size(1) != G * K || a.size(2) != off.size(2))) return py::none();
    for (const Tensor *t : {&x, &off, &w})
        for (int64_t v : t->sizes())
            if (v < 1 || v >= lim) return py::none();
    d2c_conv1d_desc q;
    std::memset(&q, 0, sizeof q);
    q.N = (int)x.size(0); q.Cin = (int)x.size(1); q.Cout = (int)w.size(0); q.L = (int)x.size(2); q.k = (int)K;
    q.s = (int)s; q.p = (int)p; q.d = (int)d; q.groups = (int)groups; q.offset_groups = (int)G; q.Lo = (int)off.size(2);
    q.dtype = dt; q.aux_dtype = adt; q.reference_quirks = quirks ? 1 : 0;
    check(d2c_conv1d_check(&q), "deform_conv1d");
    const bool grad = wants_grad(x, off, a, w, b);
    std::shared_ptr<DeformConv1dBackward> node;
    if (grad) {
        node = std::shared_ptr<DeformConv1dBackward>(new DeformConv1dBackward(), torch::autograd::deleteNode);
        node->set_next_edges(torch::autograd::collect_next_edges(x, off, a, w, b));
    }
    Tensor out;
    {
        c10::DeviceGuard guard(dev);
        const hipStream_t st = stream_of(x);
        out = at::empty({q.N, q.Cout, q.Lo}, x.options().requires_grad(false));
        const size_t nb = d2c_conv1d_forward_workspace_bytes(&q);
        const Tensor ws = workspace(nb, x, st);
        check(d2c_conv1d_forward(&q, ptr(x), ptr(off), ptr(a), ptr(w), ptr(b), ptr(out), ptr(ws), nb, st), "deform_conv1d forward");
    }
    if (!grad) return py::cast(out);
    node->q = q;
    node->x = SavedVariable(x, false); node->off = SavedVariable(off, false); node->w = SavedVariable(w, false);
    node->has_alpha = a.defined(); node->has_bias = b.defined();
    if (a.defined()) node->alpha = SavedVariable(a, false);
    return py::cast(record(out, node));
}

// ---------------------------------------------------------------- the ordinary convolution of a deformation branch
struct PlainConv3dBackward : public Node {
    d2c_conv3d_desc q;
    SavedVariable kept, w;           // the input channels-last, as the forward call made it
    bool has_bias = false;
    std::string name() const override { return "PlainConv3dBackward"; }
    void release_variables() override
    {
        const std::lock_guard<std::mutex> lock(mutex_);
        w.reset_data(); kept.reset_data();
    }
    variable_list apply(variable_list &&grads) override
    {
        variable_list r(3);
        const std::lock_guard<std::mutex> lock(mutex_);
        if (!grads[0].defined()) grads[0] = input_metadata(0).zeros_like();
        {
            at::NoGradGuard no_grad;
            const Tensor vw = w.unpack(), copy = kept.unpack();
            c10::DeviceGuard guard(vw.device());
            const hipStream_t st = stream_of(vw);
            const Tensor g = grads[0].contiguous();
            const auto opt = vw.options().requires_grad(false);
            if (should_compute_output(0)) r[0] = at::empty({q.N, q.Cin, q.D, q.H, q.W}, opt);
            if (should_compute_output(1)) r[1] = no_grad_empty_like(vw);
            if (has_bias && should_compute_output(2)) r[2] = at::empty({q.Cout}, opt);
            const size_t nb = d2c_plain_conv3d_backward_workspace_bytes(&q);
            const Tensor ws = workspace(nb, vw, st);
            check(d2c_plain_conv3d_backward(&q, ptr(g), ptr(copy), copy.numel(), ptr(vw), ptr(r[0]), ptr(r[1]), ptr(r[2]), ptr(ws), nb, st),
                  "plain_conv3d backward");
        }
        once_differentiable(r, grads[0]);
        return r;
    }
};

py::object plain_conv3d(const Tensor &x, const Tensor &w, const opt_tensor &bias, int3_t s, int3_t p, int3_t d)
{
    const Tensor b = bias.value_or(Tensor());
    if (!plain(x) || !plain(w) || (b.defined() && !plain(b)) || x.dim() != 5 || w.dim() != 5 || (b.defined() && b.dim() != 1)) return py::none();
    if (w.device() != x.device() || (b.defined() && b.device() != x.device())) return py::none();
    if (x.scalar_type() != at::kBFloat16 || w.scalar_type() != at::kBFloat16 || (b.defined() && b.scalar_type() != at::kBFloat16)) return py::none();
    if (w.size(1) != x.size(1) || (b.defined() && b.size(0) != w.size(0))) return py::none();
    d2c_conv3d_desc q;
    std::memset(&q, 0, sizeof q);
    int out_dims[3];
    for (int i = 0; i < 3; i++) {
        if (s[i] < 1 || d[i] < 1) return py::none();
        const int64_t span = x.size(2 + i) + 2 * p[i] - (d[i] * (w.size(2 + i) - 1) + 1);
        if (span < 0 || x.size(2 + i) >= (1ll << 31)) return py::none();
        out_dims[i] = (int)(span / s[i]) + 1;
    }
    q.N = (int)x.size(0); q.Cin = (int)x.size(1); q.Cout = (int)w.size(0);
    q.D = (int)x.size(2); q.H = (int)x.size(3); q.W = (int)x.size(4);
    q.kd = (int)w.size(2); q.kh = (int)w.size(3); q.kw = (int)w.size(4);
    q.sd = s[0]; q.sh = s[1]; q.sw = s[2]; q.pd = p[0]; q.ph = p[1]; q.pw = p[2]; q.dd = d[0]; q.dh = d[1]; q.dw = d[2];
    q.groups = q.offset_groups = 1;
    q.Do = out_dims[0]; q.Ho = out_dims[1]; q.Wo = out_dims[2];
    q.dtype = q.aux_dtype = D2C_BF16;
    q.epilogue_scale = 1.f;
    const size_t nc = d2c_plain_conv3d_input_bytes(&q);
    if (nc == 0) return py::none();
    const bool grad = wants_grad(x, w, b);
    std::shared_ptr<PlainConv3dBackward> node;
    if (grad) {
        node = std::shared_ptr<PlainConv3dBackward>(new PlainConv3dBackward(), torch::autograd::deleteNode);
        node->set_next_edges(torch::autograd::collect_next_edges(x, w, b));
    }
    c10::DeviceGuard guard(x.device());
    const hipStream_t st = stream_of(x);
    Tensor out = at::empty({q.N, q.Cout, q.Do, q.Ho, q.Wo}, x.options().requires_grad(false));
    const Tensor copy = at::empty({(int64_t)nc}, x.options().dtype(at::kByte).requires_grad(false));
    const size_t nb = d2c_plain_conv3d_forward_workspace_bytes(&q);
    const Tensor ws = workspace(nb, x, st);
    check(d2c_plain_conv3d_forward(&q, ptr(x), ptr(w), ptr(b), ptr(out), ptr(copy), nc, ptr(ws), nb, st), "plain_conv3d forward");
    if (!grad) return py::cast(out);
    node->q = q;
    node->kept = SavedVariable(copy, false);
    node->w = SavedVariable(w, false);
    node->has_bias = b.defined();
    return py::cast(record(out, node));
}

// ---------------------------------------------------------------- depthwise_separable_conv3d
struct DepthwiseConv3dBackward : public Node {
    d2c_dwconv3d_desc q;
    SavedVariable x, w;
    bool has_bias = false;
    std::string name() const override { return "DepthwiseConv3dBackward"; }
    void release_variables() override
    {
        const std::lock_guard<std::mutex> lock(mutex_);
        x.reset_data(); w.reset_data();
    }
    variable_list apply(variable_list &&grads) override
    {
        variable_list r(3);
        const std::lock_guard<std::mutex> lock(mutex_);
        if (!grads[0].defined()) grads[0] = input_metadata(0).zeros_like();
        {
            at::NoGradGuard no_grad;
            const Tensor vx = x.unpack(), vw = w.unpack();
            c10::DeviceGuard guard(vx.device());
            const hipStream_t st = stream_of(vx);
            const Tensor g = grads[0].contiguous();
            const bool want_w = should_compute_output(1), want_b = has_bias && should_compute_output(2);
            if (should_compute_output(0)) r[0] = no_grad_empty_like(vx);
            if (want_w) r[1] = no_grad_empty_like(vw);
            if (want_b) r[2] = at::empty({q.Cout}, vw.options().requires_grad(false));
            const size_t nb = want_w || want_b ? d2c_dwconv3d_backward_workspace_bytes(&q) : 0;
            const Tensor ws = workspace(nb, vx, st);
            check(d2c_dwconv3d_backward(&q, ptr(g), ptr(vx), ptr(vw), ptr(r[0]), ptr(r[1]), ptr(r[2]), ptr(ws), nb, st),
                  "depthwise_separable_conv3d backward");
        }
        return r;
    }
};

py::object dwconv3d(const Tensor &x, const Tensor &w, const opt_tensor &bias, int3_t s, int3_t p, int3_t d)
{
    const Tensor b = bias.value_or(Tensor());
    if (!plain(x) || !plain(w) || (b.defined() && !plain(b)) || x.dim() != 5 || w.dim() != 5 || (b.defined() && b.dim() != 1)) return py::none();
    if (w.device() != x.device() || (b.defined() && b.device() != x.device())) return py::none();
    const int dt = dtype_code(x);
    if (dt < 0 || dtype_code(w) != dt || (b.defined() && (dtype_code(b) != dt || b.size(0) != w.size(0))) || w.size(1) != 1) return py::none();
    d2c_dwconv3d_desc q;
    std::memset(&q, 0, sizeof q);
    int out_dims[3];
    for (int i = 0; i < 3; i++) {
        if (s[i] < 1 || p[i] < 0 || d[i] < 1 || x.size(2 + i) >= (1ll << 31)) return py::none();
        const int64_t span = x.size(2 + i) + 2 * p[i] - (d[i] * (w.size(2 + i) - 1) + 1);
        if (span < 0) return py::none();
        out_dims[i] = (int)(span / s[i]) + 1;
    }
    q.N = (int)x.size(0); q.C = (int)x.size(1); q.Cout = (int)w.size(0);
    q.D = (int)x.size(2); q.H = (int)x.size(3); q.W = (int)x.size(4);
    q.kd = (int)w.size(2); q.kh = (int)w.size(3); q.kw = (int)w.size(4);
    q.sd = s[0]; q.sh = s[1]; q.sw = s[2]; q.pd = p[0]; q.ph = p[1]; q.pw = p[2]; q.dd = d[0]; q.dh = d[1]; q.dw = d[2];
    q.Do = out_dims[0]; q.Ho = out_dims[1]; q.Wo = out_dims[2];
    q.dtype = dt;
    if (d2c_dwconv3d_check(&q) != D2C_OK) return py::none();
    const bool grad = wants_grad(x, w, b);
    std::shared_ptr<DepthwiseConv3dBackward> node;
    if (grad) {
        node = std::shared_ptr<DepthwiseConv3dBackward>(new DepthwiseConv3dBackward(), torch::autograd::deleteNode);
        node->set_next_edges(torch::autograd::collect_next_edges(x, w, b));
    }
    Tensor out;
    {
        c10::DeviceGuard guard(x.device());
        out = at::empty({q.N, q.Cout, q.Do, q.Ho, q.Wo}, x.options().requires_grad(false));
        check(d2c_dwconv3d_forward(&q, ptr(x), ptr(w), ptr(b), ptr(out), stream_of(x)), "depthwise_separable_conv3d");
    }
    if (!grad) return py::cast(out);
    node->q = q;
    node->x = SavedVariable(x, false); node->w = SavedVariable(w, false);
    node->has_bias = b.defined();
    return py::cast(record(out, node));
}

}  // namespace

PYBIND11_MODULE(_native, m)
{
    m.def("init", [](py::dict cache, py::list on, py::object make) {
        g_ws_cache = cache.release().ptr(); g_ws_on = on.release().ptr(); g_ws_make = make.release().ptr();
    });
    m.def("conv3d", &conv3d);
    m.def("conv3d_sized", &conv3d_sized);
    m.def("conv3d_packed", &conv3d_packed);
    m.def("conv1d", &conv1d);
    m.def("plain_conv3d", &plain_conv3d);
    m.def("dwconv3d", &dwconv3d);
}
