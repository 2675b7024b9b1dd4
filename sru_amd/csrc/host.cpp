// The host side of a call in native code: what functional.py does between torch tensors and the C ABI,
// for the plain case only (a contiguous, aligned, already converted set of tensors on one device, the
// state kept as checkpoints or not at all). Every function answers None where anything is out of the
// ordinary, before it has launched anything, and functional.py then goes its general way, which also
// says what is wrong with a call. No state is kept between calls.
//
// Why: a forward and backward pass of the recurrence cost the host 145-175 us in Python, more than the
// kernels of most sizes take. 128 x 32 x 1024 f32 with padding, 53 us of kernels: 159 us a pass then,
// 90-94 us through here (the rest is torch's own autograd); one token through ten layers of 2048: 221
// and 133 us.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <ATen/ATen.h>
#include <ATen/PythonTorchFunctionTLS.h>
#include <ATen/autocast_mode.h>
#include <c10/core/DeviceGuard.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/PyInterpreter.h>
#include <torch/csrc/autograd/python_variable.h>

#include "sru_amd.h"

namespace {

// An argument that has to be a tensor or None.
struct Arg {
    const at::Tensor *t = nullptr;   // null: None
    explicit operator bool() const { return t != nullptr; }
    const at::Tensor *operator->() const { return t; }
    void *ptr() const { return t ? t->data_ptr() : nullptr; }
};
// (a tensor of torch's own types: what a subclass holds is its own business, as are tensors without memory)
bool read(PyObject *o, Arg &a) {
    if (o == Py_None) return true;
    if (!THPVariable_CheckExact(o)) return false;
    a.t = &THPVariable_Unpack(o);
    return a->defined() && a->layout() == at::kStrided && a->has_storage();
}
// Whether a mode sees every call of torch (an operation counter, say): then all of them are made in Python.
// The mode behind `with torch.device(...)` and torch.set_default_device only places tensors that name no
// device, of which there are none here.
PyObject *device_context = nullptr;   // its class
bool observed() {
    if (c10::impl::dispatch_mode_enabled()) return true;
    if (!at::impl::torch_function_mode_enabled()) return false;
    using Modes = at::impl::PythonTorchFunctionTLS;
    for (int64_t i = 0; i < Modes::stack_len(); ++i)
        if (reinterpret_cast<PyObject *>(Py_TYPE(Modes::get_stack_at(i)->ptr(getPyInterpreter()))) != device_context) return true;
    return false;
}
bool read(PyObject *o, int64_t &v) {
    if (!PyLong_Check(o)) return false;
    v = PyLong_AsLongLong(o);
    if (v == -1 && PyErr_Occurred()) {
        PyErr_Clear();
        return false;
    }
    return true;
}
// (an argument without a truth value is for the general way to refuse)
bool read(PyObject *o, bool &v) {
    const int truth = PyObject_IsTrue(o);
    if (truth < 0) PyErr_Clear();
    v = truth == 1;
    return truth >= 0;
}

bool aligned(const at::Tensor &t, uintptr_t n) { return reinterpret_cast<uintptr_t>(t.data_ptr()) % n == 0; }
bool narrow(at::ScalarType t) { return t == at::kHalf || t == at::kBFloat16; }

// contiguous, on the device of the call, so many elements, so aligned
bool plain(const at::Tensor &t, const c10::Device &device, int64_t numel, uintptr_t alignment) {
    return t.device() == device && t.numel() == numel && t.is_contiguous() && !t.is_conj() && !t.is_neg() && aligned(t, alignment);
}

// A small tensor as the kernels read it: float, or (where `may_narrow`) in the 16-bit stream type.
bool small(const Arg &a, const c10::Device &device, int64_t numel, at::ScalarType stream, bool may_narrow, uint32_t bit, uint32_t &small16) {
    if (!a) return true;
    if (may_narrow && narrow(stream) && a->scalar_type() == stream) {
        small16 |= bit;
        return plain(*a.t, device, numel, 2);
    }
    return a->scalar_type() == at::kFloat && plain(*a.t, device, numel, 8);
}

struct Call {
    Arg u, x, weight_c, bias, init, scale, mask_c, pad;
    int64_t act = 0, d = 0, length = 0, batch = 0;
    bool bidirectional = false, has_skip = false;
    sru_amd_shape shape{};
    uint32_t small16 = 0;
    int64_t width() const { return shape.hidden * shape.dirs; }
    const c10::Device device() const { return u->device(); }
};

bool dtype_code(at::ScalarType t, int32_t &code) {
    code = t == at::kFloat ? SRU_AMD_F32 : t == at::kHalf ? SRU_AMD_F16 : SRU_AMD_BF16;
    return t == at::kFloat || narrow(t);
}

bool plain_pad(const Arg &pad, const c10::Device &device, int64_t length, int64_t batch) {
    return !pad || (pad->scalar_type() == at::kBool && pad->dim() == 2 && pad->size(0) == length && pad->size(1) == batch &&
                    plain(*pad.t, device, length * batch, 1));
}

// Sizes and flags as _Problem derives them, and the checks of _prepare_inputs; length and batch are set.
bool prepare(Call &c, bool checkpointed, bool may_narrow) {
    if (!c.u || !c.weight_c || !c.bias || !c.u->is_cuda() || c.u->dim() < 1 || c.length < 1 || c.batch < 1 || c.d < 1) return false;
    const at::ScalarType type = c.u->scalar_type();
    const c10::Device device = c.u->device();
    sru_amd_shape &s = c.shape;
    if (!dtype_code(type, s.dtype) || c.weight_c->dim() != 1 || (c.act != 0 && c.act != 1)) return false;
    s.length = c.length;
    s.batch = c.batch;
    s.hidden = c.d;
    s.dirs = c.bidirectional ? 2 : 1;
    const int64_t width = c.d * s.dirs, streams = c.u->size(-1) / width;
    if ((streams != 3 && streams != 4) || c.u->size(-1) != streams * width) return false;
    s.k = (int32_t)streams;
    s.activation_type = (int32_t)c.act;
    s.skip_type = !c.has_skip ? 0 : s.k == 3 ? 1 : 2;
    s.is_custom = 0;
    const int64_t cells = c.length * c.batch * width;
    if (checkpointed && ((type != at::kFloat && c.d % 2 != 0) || (s.skip_type == 0 && s.k == 4))) return false;
    s.state_interval = checkpointed ? SRU_AMD_STATE_INTERVAL : 1;
    s.x_dtype = SRU_AMD_X_AS_STREAMS;
    if (!plain(*c.u.t, device, cells * s.k, 16)) return false;
    if (s.skip_type == 1) {
        if (!c.x || !plain(*c.x.t, device, cells, 4)) return false;
        if (c.x->scalar_type() != type) {
            if (c.x->scalar_type() != at::kFloat || c.act != 0 || c.d % 2 != 0) return false;
            s.x_dtype = SRU_AMD_X_F32;
        }
    } else {
        c.x = Arg{};
        c.scale = Arg{};
    }
    return small(c.weight_c, device, 2 * width, type, may_narrow, SRU_AMD_SMALL_WEIGHT_C, c.small16) &&
           small(c.bias, device, 2 * width, type, may_narrow, SRU_AMD_SMALL_BIAS, c.small16) &&
           small(c.init, device, c.batch * width, type, may_narrow, SRU_AMD_SMALL_INIT, c.small16) &&
           small(c.scale, device, 1, type, may_narrow, SRU_AMD_SMALL_SCALE, c.small16) &&
           small(c.mask_c, device, c.batch * width, type, may_narrow, SRU_AMD_SMALL_MASK, c.small16) &&
           plain_pad(c.pad, device, c.length, c.batch);
}

void *stream_of(const c10::Device &device) { return c10::hip::getCurrentHIPStream(device.index()).stream(); }

// Other Python threads run while this one allocates, multiplies and launches, each of which may wait (for
// memory, for room in a queue), as they do in torch's own calls. The tensors are held by the caller's arguments.
class Unlocked {
    PyThreadState *const state = PyEval_SaveThread();

public:
    Unlocked() = default;
    Unlocked(const Unlocked &) = delete;
    ~Unlocked() { PyEval_RestoreThread(state); }
};

PyObject *none() { Py_RETURN_NONE; }
PyObject *wrap(const at::Tensor &t) {
    if (!t.defined()) return none();
    return THPVariable_Wrap(t);
}

// scan_forward(u, x, weight_c, bias, init, act, d, bidirectional, has_skip, scale, mask_c, mask_pad, train)
//   -> (h, last, checkpoints or None, whether x and scale are read)
PyObject *scan_forward(PyObject *, PyObject *const *a, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    Call c;
    if (observed() || n != 13 || !read(a[0], c.u) || !read(a[1], c.x) || !read(a[2], c.weight_c) || !read(a[3], c.bias) || !read(a[4], c.init) ||
        !read(a[5], c.act) || !read(a[6], c.d) || !read(a[9], c.scale) || !read(a[10], c.mask_c) || !read(a[11], c.pad) ||
        !read(a[7], c.bidirectional) || !read(a[8], c.has_skip))
        return none();
    const bool train = a[12] == Py_True;
    if (!c.x || c.x->dim() != 3) return none();
    c.length = c.x->size(0);
    c.batch = c.x->size(1);
    if (!prepare(c, train, !train)) return none();
    if (narrow(c.u->scalar_type())) c.small16 |= SRU_AMD_SMALL_LAST;
    at::Tensor h, last, kept;
    int rc;
    {
        const Unlocked unlocked;
        const c10::DeviceGuard guard(c.device());
        const auto options = c.u->options();
        h = at::empty({c.length, c.batch, c.width()}, options);
        last = at::empty({c.batch, c.width()}, options);
        if (train)
            kept = at::empty({(int64_t)sru_amd_state_bytes(&c.shape) / (4 * c.batch * c.width()), c.batch, c.width()}, options.dtype(at::kFloat));
        rc = sru_amd_forward_small(&c.shape, c.small16, c.u.ptr(), c.x.ptr(), c.weight_c.ptr(), c.bias.ptr(), c.init.ptr(), c.mask_c.ptr(),
                                   static_cast<const uint8_t *>(c.pad.ptr()), c.scale.ptr(), h.data_ptr(), train ? kept.data_ptr() : nullptr,
                                   last.data_ptr(), stream_of(c.device()));
    }
    if (rc != SRU_AMD_OK) return none();
    return Py_BuildValue("(NNNO)", wrap(h), wrap(last), wrap(kept), c.shape.skip_type == 1 ? Py_True : Py_False);
    END_HANDLE_TH_ERRORS
}

// scan_backward(u, x, weight_c, bias, init, scale, mask_c, mask_pad, checkpoints, grad_h, grad_last,
//               act, d, bidirectional, has_skip, length, batch) -> (grad_u, grad_x, grad_weight_c, grad_bias, grad_init)
PyObject *scan_backward(PyObject *, PyObject *const *a, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    Call c;
    Arg kept, grad_h, grad_last;
    if (observed() || n != 17 || !read(a[0], c.u) || !read(a[1], c.x) || !read(a[2], c.weight_c) || !read(a[3], c.bias) || !read(a[4], c.init) ||
        !read(a[5], c.scale) || !read(a[6], c.mask_c) || !read(a[7], c.pad) || !read(a[8], kept) || !read(a[9], grad_h) ||
        !read(a[10], grad_last) || !read(a[11], c.act) || !read(a[12], c.d) || !read(a[15], c.length) || !read(a[16], c.batch) ||
        !read(a[13], c.bidirectional) || !read(a[14], c.has_skip))
        return none();
    if (!kept || !grad_h || !prepare(c, true, false)) return none();
    const c10::Device device = c.device();
    const int64_t width = c.width(), columns = c.batch * width;
    const at::ScalarType type = c.u->scalar_type();
    if (kept->scalar_type() != at::kFloat || !plain(*kept.t, device, (int64_t)sru_amd_state_bytes(&c.shape) / 4, 4) ||
        grad_h->scalar_type() != type || !plain(*grad_h.t, device, c.length * columns, 4) ||
        !small(grad_last, device, columns, type, true, SRU_AMD_SMALL_LAST, c.small16))
        return none();
    at::Tensor grad_u, grad_x, grad_wc, grad_bias, grad_init;
    int rc;
    {
        const Unlocked unlocked;
        const c10::DeviceGuard guard(device);
        const auto floats = c.u->options().dtype(at::kFloat);
        grad_u = at::empty(c.u->sizes(), c.u->options());
        if (c.x) grad_x = at::empty(c.x->sizes(), c.x->options());
        grad_wc = at::empty({2 * width}, floats);
        grad_bias = at::empty(c.bias->sizes(), floats);
        const int64_t need = (int64_t)sru_amd_backward_workspace_bytes(&c.shape);
        // (the gradient of an initial state that was not given is written behind the workspace)
        const at::Tensor workspace = at::empty({need / 4 + (c.init ? 0 : columns)}, floats);
        if (c.init) grad_init = at::empty(c.init->sizes(), floats);
        float *const init_out = c.init ? grad_init.data_ptr<float>() : workspace.data_ptr<float>() + need / 4;
        rc = sru_amd_backward_small(
            &c.shape, c.small16, c.u.ptr(), c.x.ptr(), c.weight_c.ptr(), c.bias.ptr(), c.init.ptr(), c.mask_c.ptr(),
            static_cast<const uint8_t *>(c.pad.ptr()), c.scale.ptr(), kept.ptr(), grad_h.ptr(), grad_last.ptr(), grad_u.data_ptr(),
            c.x ? grad_x.data_ptr() : nullptr, grad_wc.data_ptr(), grad_bias.data_ptr(), init_out, workspace.data_ptr(), (size_t)need,
            stream_of(device));
    }
    if (rc != SRU_AMD_OK) return none();
    return Py_BuildValue("(NNNNN)", wrap(grad_u), wrap(grad_x), wrap(grad_wc), wrap(grad_bias), wrap(grad_init));
    END_HANDLE_TH_ERRORS
}

// x weight, with `own` by a kernel where that is the faster one (the device is set)
at::Tensor product(const at::Tensor &x, const at::Tensor &weight, int32_t dtype, bool own) {
    const int64_t rows = x.size(0), inner = x.size(1), cols = weight.size(1);
    if (own && sru_amd_product_wanted(dtype, rows, inner, cols)) {
        at::Tensor out = at::empty({rows, cols}, x.options());
        if (sru_amd_product(dtype, rows, inner, cols, x.data_ptr(), weight.data_ptr(), out.data_ptr(), stream_of(x.device())) == SRU_AMD_OK) return out;
    }
    return at::mm(x, weight);
}

// layer_forward(x, residual, weight_proj, weight, weight_c, bias, init, act, d, bidirectional, has_skip, scale, mask_pad)
//   -> (h, last), False where no kernel takes the layer or a mode watches, None where the general way has to look
PyObject *layer_forward(PyObject *, PyObject *const *a, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    if (observed()) Py_RETURN_FALSE;   // the products are calls of their own
    Arg x, residual, weight_proj, weight, weight_c, bias, init, scale, pad;
    int64_t act = 0, d = 0;
    bool bidirectional = false, has_skip = false;
    if (n != 13 || !read(a[0], x) || !read(a[1], residual) || !read(a[2], weight_proj) || !read(a[3], weight) || !read(a[4], weight_c) ||
        !read(a[5], bias) || !read(a[6], init) || !read(a[7], act) || !read(a[8], d) || !read(a[11], scale) || !read(a[12], pad) ||
        !read(a[9], bidirectional) || !read(a[10], has_skip))
        return none();
    if (!x || !residual || !weight || !weight_c || !bias || !x->is_cuda() || x->dim() != 3 || d < 1) return none();
    const at::ScalarType type = x->scalar_type();
    if (!narrow(type)) Py_RETURN_FALSE;
    const c10::Device device = x->device();
    const int64_t length = x->size(0), batch = x->size(1), in = x->size(2), rows = length * batch;
    const int64_t dirs = bidirectional ? 2 : 1, width = d * dirs;
    int64_t inner = in;
    for (const Arg *w : {&weight_proj, &weight}) {
        if (!*w) continue;
        if ((*w)->scalar_type() != type || (*w)->dim() != 2 || (*w)->size(0) != inner || !plain(*w->t, device, (*w)->numel(), 16)) return none();
        inner = (*w)->size(1);
    }
    const int64_t n_proj = weight_proj ? weight_proj->size(1) : 0, k = inner / width;
    if ((k != 3 && k != 4) || inner != k * width || rows < 1 || weight_c->dim() != 1) return none();
    sru_amd_shape s{};
    s.length = length;
    s.batch = batch;
    s.hidden = d;
    s.dirs = (int32_t)dirs;
    s.k = (int32_t)k;
    s.activation_type = (int32_t)act;
    s.skip_type = !has_skip ? 0 : k == 3 ? 1 : 2;
    dtype_code(type, s.dtype);
    s.state_interval = 1;
    s.x_dtype = SRU_AMD_X_AS_STREAMS;
    // Both products in kernels, or the second one with the recurrence, or products and the scan: the last where
    // one of the products is a kernel (one step in 16 bits has the step kernels instead), and for one step at sizes
    // past the step kernels', where the host's time counts (4096 features, 16 rows: 29.9 us a layer, 29.7 of them
    // kernels).
    const bool whole = sru_amd_layer_route(&s, in, n_proj) != 0;
    const bool fused = whole || (n_proj && sru_amd_layer_route(&s, n_proj, 0) != 0);
    const bool own = !fused && length > 1 &&
                     (sru_amd_product_wanted(s.dtype, rows, n_proj ? n_proj : in, k * width) || (n_proj && sru_amd_product_wanted(s.dtype, rows, in, n_proj)));
    if (!fused && !own && !(length == 1 && batch <= 64 && width % 32 == 0 && in % 32 == 0 && n_proj % 32 == 0)) Py_RETURN_FALSE;
    uint32_t small16 = SRU_AMD_SMALL_LAST;
    if (s.skip_type != 1) scale = Arg{};
    if (!plain(*x.t, device, rows * in, 16) ||
        (s.skip_type == 1 && (residual->scalar_type() != type || !plain(*residual.t, device, rows * width, 16))) ||
        !small(weight_c, device, 2 * width, type, true, SRU_AMD_SMALL_WEIGHT_C, small16) ||
        !small(bias, device, 2 * width, type, true, SRU_AMD_SMALL_BIAS, small16) ||
        !small(init, device, batch * width, type, true, SRU_AMD_SMALL_INIT, small16) ||
        !small(scale, device, 1, type, true, SRU_AMD_SMALL_SCALE, small16) || !plain_pad(pad, device, length, batch))
        return none();
    at::Tensor h, last;
    int rc;
    {
        const Unlocked unlocked;
        const c10::DeviceGuard guard(device);
        const auto options = x->options();
        at::Tensor y = x->view({rows, in}), projected;
        if (n_proj && !whole) y = product(y, *weight_proj.t, s.dtype, own);
        if (n_proj && whole) projected = at::empty({rows, n_proj}, options);   // the projection is the kernels' business
        h = at::empty({length, batch, width}, options);
        last = at::empty({batch, width}, options);
        const void *const skip = s.skip_type == 1 ? residual.ptr() : nullptr;
        const uint8_t *const mask = static_cast<const uint8_t *>(pad.ptr());
        if (fused)
            rc = sru_amd_layer_forward(&s, small16, y.size(1), whole ? n_proj : 0, y.data_ptr(), skip, whole ? weight_proj.ptr() : nullptr,
                                       weight.ptr(), weight_c.ptr(), bias.ptr(), init.ptr(), mask, scale.ptr(),
                                       projected.defined() ? projected.data_ptr() : nullptr, h.data_ptr(), last.data_ptr(), stream_of(device));
        else
            rc = sru_amd_forward_small(&s, small16, product(y, *weight.t, s.dtype, own).data_ptr(), skip, weight_c.ptr(), bias.ptr(), init.ptr(), nullptr,
                                       mask, scale.ptr(), h.data_ptr(), nullptr, last.data_ptr(), stream_of(device));
    }
    if (rc != SRU_AMD_OK) return none();
    return Py_BuildValue("(NN)", wrap(h), wrap(last));
    END_HANDLE_TH_ERRORS
}

// What a cell holds under a name, borrowed; null: nothing.
struct Cell {
    PyObject *const attributes, *const parameters, *const buffers;
    static PyObject *item(PyObject *dict, const char *name) {
        PyObject *const o = dict ? PyDict_GetItemString(dict, name) : nullptr;
        return o;
    }
    explicit Cell(PyObject *dict) : attributes(dict), parameters(item(dict, "_parameters")), buffers(item(dict, "_buffers")) {}
    PyObject *attribute(const char *name) const { return item(attributes, name); }
    bool is(const char *name, PyObject *value) const { return attribute(name) == value; }
    bool number(const char *name, int64_t &v) const {
        PyObject *const o = attribute(name);
        return o && o != Py_None && read(o, v);
    }
    bool positive(const char *name) const {   // (or not a number)
        PyObject *const o = attribute(name);
        return !o || !PyFloat_Check(o) || PyFloat_AS_DOUBLE(o) != 0.0;
    }
    bool empty(const char *name) const {
        PyObject *const o = attribute(name);
        return o && PyDict_Check(o) && PyDict_GET_SIZE(o) == 0;
    }
    bool tensor(PyObject *dict, const char *name, Arg &a) const {
        PyObject *const o = item(dict, name);
        return o && read(o, a);
    }
};

// stack_forward(cells, type of a cell, x, c0, mask_pad) -> (h, last states), or None where the layers have to be called one
// by one: one of them is not of that type, has a step of its own, hooks, a normalisation, a module or dropout, or differs from the others
// in its form, or there is no kernel for the stack
PyObject *stack_forward(PyObject *, PyObject *const *a, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    Arg x, init, pad;
    if (n != 5 || !PyList_Check(a[0]) || observed() || !read(a[2], x) || !read(a[3], init) || !read(a[4], pad) || !x || !x->is_cuda() || x->dim() != 3 ||
        !narrow(x->scalar_type()))
        return none();
    const int64_t layers = PyList_GET_SIZE(a[0]), length = x->size(0), batch = x->size(1), width = x->size(2);
    constexpr int kLayers = SRU_AMD_STACK_MAX_LAYERS;
    if (layers < 1 || layers > kLayers) return none();
    const at::ScalarType type = x->scalar_type();
    const c10::Device device = x->device();
    sru_amd_shape s{};
    s.length = length;
    s.batch = batch;
    s.k = 3;
    dtype_code(type, s.dtype);
    s.state_interval = 1;
    s.x_dtype = SRU_AMD_X_AS_STREAMS;
    const void *projs[kLayers], *weights[kLayers], *wcs[kLayers], *biases[kLayers], *scales[kLayers];
    size_t need = 0;
    int64_t n_proj = 0;
    uint32_t flags = 0;
    for (int64_t l = 0; l < layers; ++l) {
        PyObject *const o = PyList_GET_ITEM(a[0], l);
        PyObject **const dict = (PyObject *)Py_TYPE(o) == a[1] ? _PyObject_GetDictPtr(o) : nullptr;
        if (!dict || !*dict) return none();
        const Cell cell(*dict);
        for (const char *own : {"forward", "compute_UV", "compute_U", "apply_recurrence", "_whole_layer", "_normalise", "_call_impl", "_compiled_call_impl"})
            if (cell.attribute(own)) return none();
        for (const char *hooks : {"_forward_hooks", "_forward_pre_hooks", "_backward_hooks", "_backward_pre_hooks"})
            if (!cell.empty(hooks)) return none();
        PyObject *const native = cell.attribute("native_16bit");
        if (!cell.is("custom_m", Py_None) || !cell.is("layer_norm", Py_None) || (native && native != Py_True) ||
            (!cell.is("training", Py_False) && (cell.positive("dropout") || cell.positive("rnn_dropout"))))
            return none();
        int64_t d = 0, act = 0, inputs = 0;
        bool both = false, has_skip = false, rescale = false;
        if (!cell.number("hidden_size", d) || !cell.number("activation_type", act) || !cell.number("input_size", inputs) || !cell.attribute("bidirectional") ||
            !cell.attribute("has_skip_term") || !cell.attribute("rescale") || !read(cell.attribute("bidirectional"), both) ||
            !read(cell.attribute("has_skip_term"), has_skip) || !read(cell.attribute("rescale"), rescale))
            return none();
        Arg proj, weight, weight_c, bias, scale;
        if (!cell.tensor(cell.parameters, "weight", weight) || !cell.tensor(cell.parameters, "weight_c", weight_c) || !cell.tensor(cell.parameters, "bias", bias) ||
            !(cell.tensor(cell.parameters, "weight_proj", proj) || cell.is("weight_proj", Py_None)) || !weight || !weight_c || !bias)
            return none();
        if (rescale && !cell.tensor(cell.buffers, "scale_x", scale)) return none();
        const int64_t project = proj ? (proj->dim() == 2 ? proj->size(1) : -1) : 0;
        if (l == 0) {
            s.hidden = d;
            s.dirs = both ? 2 : 1;
            s.activation_type = (int32_t)act;
            s.skip_type = has_skip ? 1 : 0;
            n_proj = project;
            if (d < 1 || d * s.dirs != width || (act != 0 && act != 1)) return none();
            need = sru_amd_stack_workspace_bytes(&s, layers, n_proj);
            if (need == 0) return none();
        }
        const int64_t inner = n_proj ? n_proj : width;
        uint32_t small16 = 0;
        if (d != s.hidden || (both ? 2 : 1) != s.dirs || act != s.activation_type || has_skip != (s.skip_type == 1) || project != n_proj || inputs != width ||
            weight->scalar_type() != type || weight->dim() != 2 || weight->size(0) != inner || weight->size(1) != 3 * width || !plain(*weight.t, device, inner * 3 * width, 16) ||
            (proj && (proj->scalar_type() != type || proj->size(0) != width || !plain(*proj.t, device, width * n_proj, 16))) || weight_c->dim() != 1 ||
            !small(weight_c, device, 2 * width, type, true, SRU_AMD_SMALL_WEIGHT_C, small16) ||
            !small(bias, device, 2 * width, type, true, SRU_AMD_SMALL_BIAS, small16) || !small(scale, device, 1, type, true, SRU_AMD_SMALL_SCALE, small16))
            return none();
        if (!scale) small16 |= flags & SRU_AMD_SMALL_SCALE;
        if (l == 0) flags = small16;
        if (small16 != flags) return none();
        projs[l] = proj.ptr();
        weights[l] = weight.ptr();
        wcs[l] = weight_c.ptr();
        biases[l] = bias.ptr();
        scales[l] = s.skip_type == 1 ? scale.ptr() : nullptr;
    }
    if (!plain(*x.t, device, length * batch * width, 16) || (init && (init->dim() != 3 || init->size(0) != layers)) ||
        !small(init, device, layers * batch * width, type, true, SRU_AMD_SMALL_INIT, flags) || !plain_pad(pad, device, length, batch))
        return none();
    at::Tensor h, last;
    int rc;
    {
        const Unlocked unlocked;
        const c10::DeviceGuard guard(device);
        const auto options = x->options();
        h = at::empty({length, batch, width}, options);
        last = at::empty({layers, batch, width}, options);
        const at::Tensor workspace = at::empty({(int64_t)need / 4}, options.dtype(at::kFloat));
        rc = sru_amd_stack_forward(&s, flags | SRU_AMD_SMALL_LAST, layers, n_proj, x.ptr(), projs, weights, wcs, biases, scales, init.ptr(),
                                   static_cast<const uint8_t *>(pad.ptr()), h.data_ptr(), last.data_ptr(), workspace.data_ptr(), need, stream_of(device));
    }
    if (rc != SRU_AMD_OK) return none();
    return Py_BuildValue("(NN)", wrap(h), wrap(last));
    END_HANDLE_TH_ERRORS
}

// product(x, weight) -> x weight in float, by the kernel where that is the faster one, else None
PyObject *float_product(PyObject *, PyObject *const *a, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    Arg x, weight;
    if (observed() || n != 2 || !read(a[0], x) || !read(a[1], weight) || !x || !weight || !x->is_cuda() || x->dim() != 2 || weight->dim() != 2 ||
        x->scalar_type() != at::kFloat || weight->scalar_type() != at::kFloat || x->size(1) != weight->size(0))
        return none();
    const int64_t rows = x->size(0), inner = x->size(1), cols = weight->size(1);
    const c10::Device device = x->device();
    if (!sru_amd_product_wanted(SRU_AMD_F32, rows, inner, cols) || !plain(*x.t, device, rows * inner, 16) || !plain(*weight.t, device, inner * cols, 16))
        return none();
    at::Tensor out;
    {
        const Unlocked unlocked;
        const c10::DeviceGuard guard(device);
        out = product(*x.t, *weight.t, SRU_AMD_F32, true);
    }
    return wrap(out);
    END_HANDLE_TH_ERRORS
}

// autocast_operand(t) -> t as autocast hands it to a product: in the region's type, a parameter converted once in a region
PyObject *autocast_operand(PyObject *, PyObject *o) {
    HANDLE_TH_ERRORS
    Arg t;
    if (!read(o, t) || !t) return none();
    at::Tensor out;
    {
        const Unlocked unlocked;
        out = at::autocast::cached_cast(at::autocast::get_autocast_dtype(at::kCUDA), *t.t, at::kCUDA);
    }
    return wrap(out);
    END_HANDLE_TH_ERRORS
}

PyObject *observed_now(PyObject *, PyObject *) {
    HANDLE_TH_ERRORS
    return PyBool_FromLong(observed());
    END_HANDLE_TH_ERRORS
}

PyMethodDef methods[] = {
    {"observed", observed_now, METH_NOARGS, nullptr},
    {"autocast_operand", autocast_operand, METH_O, nullptr},
    {"product", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(float_product)), METH_FASTCALL, nullptr},
    {"scan_forward", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(scan_forward)), METH_FASTCALL, nullptr},
    {"scan_backward", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(scan_backward)), METH_FASTCALL, nullptr},
    {"layer_forward", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(layer_forward)), METH_FASTCALL, nullptr},
    {"stack_forward", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(stack_forward)), METH_FASTCALL, nullptr},
    {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_host", "Calls of the recurrence in the plain case.", -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__host() {
    if (PyObject *device = PyImport_ImportModule("torch.utils._device")) {
        device_context = PyObject_GetAttrString(device, "DeviceContext");   // (kept for good)
        Py_DECREF(device);
    }
    PyErr_Clear();   // (not found: every mode watches)
    PyObject *m = PyModule_Create(&module);
    // the release of torch whose headers this was compiled with, for the importer to compare
    if (m && PyModule_AddStringConstant(m, "torch_version", SRU_AMD_TORCH_VERSION) != 0) Py_CLEAR(m);
    return m;
}
