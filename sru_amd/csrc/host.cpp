// The host side of a call in native code: what functional.py does between torch tensors and the C ABI,
// for the plain case only (a contiguous, aligned, already converted set of tensors on one device, the
// state kept as checkpoints or not at all). Every function answers None where anything is out of the
// ordinary, before it has launched anything, and functional.py then goes its general way, which also
// says what is wrong with a call. No state is kept between calls.
//
// Why: a forward and backward pass of the recurrence cost the host 145-175 us in Python, more than the
// kernels of most sizes take. 128 x 32 x 1024 f32 with padding, 53 us of kernels: 159 us a pass then,
// 90-94 us through here with Python's autograd around it and 73 with a node of the graph that is native as
// well; one token through ten layers of 2048: 221 us, 133 and, as one call for the stack, 71.
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
#include <torch/csrc/autograd/engine.h>
#include <torch/csrc/autograd/function.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/autograd/saved_variable.h>
#include <torch/csrc/autograd/variable.h>

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

// the first twelve arguments of a recurrence's forward call
bool read_scan(PyObject *const *a, Call &c) {
    if (!read(a[0], c.u) || !read(a[1], c.x) || !read(a[2], c.weight_c) || !read(a[3], c.bias) || !read(a[4], c.init) || !read(a[5], c.act) ||
        !read(a[6], c.d) || !read(a[9], c.scale) || !read(a[10], c.mask_c) || !read(a[11], c.pad) || !read(a[7], c.bidirectional) ||
        !read(a[8], c.has_skip) || !c.x || c.x->dim() != 3)
        return false;
    c.length = c.x->size(0);
    c.batch = c.x->size(1);
    return true;
}

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
// memory, for room in a queue), as they do in torch's own calls. The tensors are held by the caller's arguments; a call
// that is given the objects which have them (stack_forward) holds their memory itself.
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

// The recurrence of a prepared call: h, last state and, to be differentiated, the checkpoints.
int run_forward(Call &c, bool train, at::Tensor &h, at::Tensor &last, at::Tensor &kept) {
    if (narrow(c.u->scalar_type())) c.small16 |= SRU_AMD_SMALL_LAST;
    const auto options = c.u->options();
    h = at::empty({c.length, c.batch, c.width()}, options);
    last = at::empty({c.batch, c.width()}, options);
    if (train)
        kept = at::empty({(int64_t)sru_amd_state_bytes(&c.shape) / (4 * c.batch * c.width()), c.batch, c.width()}, options.dtype(at::kFloat));
    return sru_amd_forward_small(&c.shape, c.small16, c.u.ptr(), c.x.ptr(), c.weight_c.ptr(), c.bias.ptr(), c.init.ptr(), c.mask_c.ptr(),
                                 static_cast<const uint8_t *>(c.pad.ptr()), c.scale.ptr(), h.data_ptr(), train ? kept.data_ptr() : nullptr,
                                 last.data_ptr(), stream_of(c.device()));
}

// What a call's gradients need besides it, in the plain case.
bool prepare_backward(Call &c, const Arg &kept, const Arg &grad_h, const Arg &grad_last) {
    if (!kept || !grad_h || !prepare(c, true, false)) return false;
    const int64_t columns = c.batch * c.width();
    return kept->scalar_type() == at::kFloat && plain(*kept.t, c.device(), (int64_t)sru_amd_state_bytes(&c.shape) / 4, 4) &&
           grad_h->scalar_type() == c.u->scalar_type() && plain(*grad_h.t, c.device(), c.length * columns, 4) &&
           small(grad_last, c.device(), columns, c.u->scalar_type(), true, SRU_AMD_SMALL_LAST, c.small16);
}

constexpr int kGradients = 5;   // of u, x, weight_c, bias and init
int run_backward(const Call &c, const Arg &kept, const Arg &grad_h, const Arg &grad_last, at::Tensor (&grads)[kGradients]) {
    const int64_t width = c.width(), columns = c.batch * width;
    const auto floats = c.u->options().dtype(at::kFloat);
    grads[0] = at::empty(c.u->sizes(), c.u->options());
    if (c.x) grads[1] = at::empty(c.x->sizes(), c.x->options());
    grads[2] = at::empty({2 * width}, floats);
    grads[3] = at::empty(c.bias->sizes(), floats);
    const int64_t need = (int64_t)sru_amd_backward_workspace_bytes(&c.shape);
    // (the gradient of an initial state that was not given is written behind the workspace)
    const at::Tensor workspace = at::empty({need / 4 + (c.init ? 0 : columns)}, floats);
    if (c.init) grads[4] = at::empty(c.init->sizes(), floats);
    float *const init_out = c.init ? grads[4].data_ptr<float>() : workspace.data_ptr<float>() + need / 4;
    return sru_amd_backward_small(
        &c.shape, c.small16, c.u.ptr(), c.x.ptr(), c.weight_c.ptr(), c.bias.ptr(), c.init.ptr(), c.mask_c.ptr(),
        static_cast<const uint8_t *>(c.pad.ptr()), c.scale.ptr(), kept.ptr(), grad_h.ptr(), grad_last.ptr(), grads[0].data_ptr(),
        c.x ? grads[1].data_ptr() : nullptr, grads[2].data_ptr(), grads[3].data_ptr(), init_out, workspace.data_ptr(), (size_t)need,
        stream_of(c.device()));
}

// scan_forward(u, x, weight_c, bias, init, act, d, bidirectional, has_skip, scale, mask_c, mask_pad, train)
//   -> (h, last, checkpoints or None, whether x and scale are read)
PyObject *scan_forward(PyObject *, PyObject *const *a, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    Call c;
    if (observed() || n != 13 || !read_scan(a, c)) return none();
    const bool train = a[12] == Py_True;
    if (!prepare(c, train, !train)) return none();
    at::Tensor h, last, kept;
    int rc;
    {
        const Unlocked unlocked;
        const c10::DeviceGuard guard(c.device());
        rc = run_forward(c, train, h, last, kept);
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
    if (!prepare_backward(c, kept, grad_h, grad_last)) return none();
    at::Tensor grads[kGradients];
    int rc;
    {
        const Unlocked unlocked;
        const c10::DeviceGuard guard(c.device());
        rc = run_backward(c, kept, grad_h, grad_last, grads);
    }
    if (rc != SRU_AMD_OK) return none();
    return Py_BuildValue("(NNNNN)", wrap(grads[0]), wrap(grads[1]), wrap(grads[2]), wrap(grads[3]), wrap(grads[4]));
    END_HANDLE_TH_ERRORS
}

// out = x weight, by a kernel where that is the faster one (the device is set)
void product_into(at::Tensor &out, const at::Tensor &x, const at::Tensor &weight, int32_t dtype) {
    const int64_t rows = x.size(0), inner = x.size(1), cols = weight.size(1);
    if (sru_amd_product_wanted(dtype, rows, inner, cols) && aligned(x, 16) && aligned(weight, 16) && weight.is_contiguous() && x.is_contiguous() &&
        sru_amd_product(dtype, rows, inner, cols, x.data_ptr(), weight.data_ptr(), out.data_ptr(), stream_of(x.device())) == SRU_AMD_OK)
        return;
    at::mm_out(out, x, weight);
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

// ---------------------------------------------------------------- autograd
// The graph's own nodes in the plain case. Python's autograd Functions cost some 25 us of host time a pass more for the
// recurrence and 60 for a layer: two float layers of 256, 32 steps of 32 rows, 320 -> 152-165 or 213-223 us a training step (the
// host takes one time or the other, by process) with 93 us of kernels; the recurrence alone, 128 x 32 x 1024 float padded, 96 -> 76 us with 53. A layer that knows both of its parts also adds the
// skip term's gradient in the product that makes the rest of it: 512 x 16 rows, ten layers of 2048 under autocast 4246 -> 4091 us.

using torch::autograd::SavedVariable;
using torch::autograd::Variable;
using torch::autograd::variable_list;

bool usable(const at::Tensor &t) {   // (what came back from a hook or from another node)
    return !t.defined() || (t.layout() == at::kStrided && t.has_storage() && !t.key_set().has(c10::DispatchKey::Python));
}

// Tensors and flags of a recurrence between its forward and backward pass.
struct Kept {
    enum { U, X, WeightC, Bias, Init, Scale, MaskC, Pad, States, kCount };
    SavedVariable saved[kCount];
    int64_t act = 0, d = 0, length = 0, batch = 0;
    bool bidirectional = false, has_skip = false;

    void keep(const Call &c, const at::Tensor &states) {
        const auto save = [](const Arg &a) { return a ? SavedVariable(*a.t, false) : SavedVariable(); };
        const Arg of_states{&states};
        int i = 0;
        for (const Arg *a : {&c.u, &c.x, &c.weight_c, &c.bias, &c.init, &c.scale, &c.mask_c, &c.pad, &of_states}) saved[i++] = save(*a);
        act = c.act;
        d = c.d;
        length = c.length;
        batch = c.batch;
        bidirectional = c.bidirectional;
        has_skip = c.has_skip;
    }
    void release() {
        for (SavedVariable &v : saved) v.reset_data();
    }
};

// functional._scan_gradients(saved tensors, call, grad_h, grad_last): the general way, and what is wrong with a call
void general_gradients(const Kept &k, const variable_list &saved, const at::Tensor &grad_h, const at::Tensor &grad_last, at::Tensor (&grads)[kGradients]) {
    struct Locked {
        const PyGILState_STATE state = PyGILState_Ensure();
        ~Locked() { PyGILState_Release(state); }
    } locked;
    const auto raise = [] {
        python_error error;
        error.persist();
        throw error;
    };
    PyObject *tensors = PyTuple_New((Py_ssize_t)saved.size());
    for (size_t i = 0; tensors && i < saved.size(); ++i) PyTuple_SET_ITEM(tensors, (Py_ssize_t)i, wrap(saved[i]));
    PyObject *const module = tensors ? PyImport_ImportModule("sru_amd.functional") : nullptr;
    PyObject *const out = module ? PyObject_CallMethod(module, "_scan_gradients", "N(LLOOLL)NN", tensors, (long long)k.act, (long long)k.d,
                                                       k.bidirectional ? Py_True : Py_False, k.has_skip ? Py_True : Py_False, (long long)k.length,
                                                       (long long)k.batch, wrap(grad_h), wrap(grad_last))
                                 : nullptr;
    Py_XDECREF(module);
    if (!out) raise();
    for (int i = 0; i < kGradients; ++i) {
        PyObject *const o = PyTuple_GET_ITEM(out, i);
        if (o != Py_None) grads[i] = THPVariable_Unpack(o);
    }
    Py_DECREF(out);
}

void gradients_of(const Kept &k, const std::shared_ptr<torch::autograd::Node> &node, const at::Tensor &grad_h, const at::Tensor &grad_last,
                  at::Tensor (&grads)[kGradients]) {
    variable_list t;
    for (const SavedVariable &v : k.saved) t.push_back(v.unpack(node));
    bool as_usual = !observed() && usable(grad_h) && usable(grad_last);
    for (const at::Tensor &v : t) as_usual = as_usual && usable(v);
    if (as_usual) {
        const auto arg = [&](const at::Tensor &v) { return Arg{v.defined() ? &v : nullptr}; };
        Call c;
        c.u = arg(t[Kept::U]);
        c.x = arg(t[Kept::X]);
        c.weight_c = arg(t[Kept::WeightC]);
        c.bias = arg(t[Kept::Bias]);
        c.init = arg(t[Kept::Init]);
        c.scale = arg(t[Kept::Scale]);
        c.mask_c = arg(t[Kept::MaskC]);
        c.pad = arg(t[Kept::Pad]);
        c.act = k.act;
        c.d = k.d;
        c.length = k.length;
        c.batch = k.batch;
        c.bidirectional = k.bidirectional;
        c.has_skip = k.has_skip;
        const Arg states = arg(t[Kept::States]), gh = arg(grad_h), gl = arg(grad_last);
        if (prepare_backward(c, states, gh, gl)) {
            const c10::DeviceGuard guard(c.device());
            if (run_backward(c, states, gh, gl, grads) == SRU_AMD_OK) return;
        }
    }
    general_gradients(k, t, grad_h, grad_last, grads);
}

struct RecurrenceNode : torch::autograd::Node {
    Kept kept;
    std::string name() const override { return "ElementwiseRecurrenceBackward"; }
    void release_variables() override {
        const std::lock_guard<std::mutex> lock(mutex_);
        kept.release();
    }
    variable_list apply(variable_list &&out) override {
        const std::lock_guard<std::mutex> lock(mutex_);
        at::Tensor grads[kGradients];
        gradients_of(kept, shared_from_this(), out[0], out[1], grads);
        return variable_list(grads, grads + kGradients);
    }
};

template <typename N> std::shared_ptr<N> new_node() { return std::shared_ptr<N>(new N(), torch::autograd::deleteNode); }
bool wants(const Arg &a) { return a && a->requires_grad(); }
Variable variable(const Arg &a) { return a ? *a.t : Variable(); }

// recurrence(u, x, weight_c, bias, init, act, d, bidirectional, has_skip, scale, mask_c, mask_pad) -> (h, last), in the graph
// where gradients are recorded, or None: not the plain case
PyObject *recurrence(PyObject *, PyObject *const *a, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    Call c;
    if (observed() || n != 12 || !read_scan(a, c)) return none();
    const Call given = c;
    if (!prepare(c, true, false)) return none();
    at::Tensor h, last, states;
    int rc;
    {
        const Unlocked unlocked;
        const c10::DeviceGuard guard(c.device());
        rc = run_forward(c, true, h, last, states);
    }
    if (rc != SRU_AMD_OK) return none();
    if (at::GradMode::is_enabled() && (wants(given.u) || wants(given.x) || wants(given.weight_c) || wants(given.bias) || wants(given.init))) {
        const auto node = new_node<RecurrenceNode>();
        node->set_next_edges(torch::autograd::collect_next_edges(variable(given.u), variable(given.x), variable(given.weight_c), variable(given.bias),
                                                                 variable(given.init)));
        node->kept.keep(c, states);
        torch::autograd::create_gradient_edge(h, node);
        torch::autograd::create_gradient_edge(last, node);
    }
    return Py_BuildValue("(NN)", wrap(h), wrap(last));
    END_HANDLE_TH_ERRORS
}

// x^T grad in `dtype` (under a mode that sees every call, or of what a hook made something else of, a call of torch's)
at::Tensor weight_gradient(const at::Tensor &x, const at::Tensor &grad, at::ScalarType dtype) {
    int32_t code = 0, out_code = 0;
    const int64_t rows = x.size(0), inner = x.size(1), cols = grad.size(1);
    if (!at::GradMode::is_enabled() && !observed() && usable(x) && usable(grad) && narrow(x.scalar_type()) && x.scalar_type() == grad.scalar_type() && dtype_code(x.scalar_type(), code) &&
        dtype_code(dtype, out_code) && plain(x, grad.device(), rows * inner, 16) && plain(grad, grad.device(), rows * cols, 16)) {
        const int64_t need = (int64_t)sru_amd_product_grad_workspace_bytes(code, rows, inner, cols);
        if (need > 0) {
            at::Tensor out = at::empty({inner, cols}, x.options().dtype(dtype));
            const at::Tensor workspace = at::empty({need / 4}, x.options().dtype(at::kFloat));
            if (sru_amd_product_grad(code, rows, inner, cols, x.data_ptr(), grad.data_ptr(), out_code, out.data_ptr(), workspace.data_ptr(),
                                     (size_t)need, stream_of(x.device())) == SRU_AMD_OK)
                return out;
        }
    }
    return at::mm(x.t(), grad).to(dtype);
}

// A layer: the dense products and the recurrence behind them. The input's gradient is the skip term's plus the product's,
// which the product adds to it where both are of one type.
struct LayerNode : torch::autograd::Node {
    enum { Input, Residual, WeightProj, Weight, WeightC, Bias, Init };
    Kept kept;
    SavedVariable operand, projected, weight_proj, weight;   // as the products read them
    at::ScalarType input_type = at::kFloat, proj_type = at::kFloat, weight_type = at::kFloat;   // as they were given
    bool one_input = false, has_proj = false;                // the skip term reads the layer's input
    std::string name() const override { return "SRULayerBackward"; }
    void release_variables() override {
        const std::lock_guard<std::mutex> lock(mutex_);
        kept.release();
        for (SavedVariable *v : {&operand, &projected, &weight_proj, &weight}) v->reset_data();
    }
    variable_list apply(variable_list &&out) override {
        const std::lock_guard<std::mutex> lock(mutex_);
        const c10::impl::ExcludeDispatchKeyGuard as_they_are(c10::autocast_dispatch_keyset);
        const auto self = shared_from_this();
        at::Tensor grads[kGradients];
        gradients_of(kept, self, out[0], out[1], grads);
        if (!torch::autograd::get_current_graph_task_keep_graph()) kept.release();   // (room for the products' results)
        const c10::DeviceGuard guard(grads[0].device());
        variable_list result(7);
        result[WeightC] = grads[2];
        result[Bias] = grads[3];
        result[Init] = grads[4];
        const int64_t rows = kept.length * kept.batch;
        at::Tensor grad = grads[0].view({rows, -1});
        const bool input = task_should_compute_output(Input), of_proj = has_proj && task_should_compute_output(WeightProj);
        const auto flat = [&](const SavedVariable &v) {
            const at::Tensor t = v.unpack(self);
            return t.reshape({rows, t.size(-1)});
        };
        if (task_should_compute_output(Weight)) {   // (to be differentiated again: as a function of what was projected)
            const at::Tensor x = !has_proj ? flat(operand) : at::GradMode::is_enabled() ? at::mm(flat(operand), weight_proj.unpack(self)) : flat(projected);
            result[Weight] = weight_gradient(x, grad, weight_type);
        }
        if (has_proj && (input || of_proj)) {
            grad = at::mm(grad, weight.unpack(self).t());
            if (of_proj) result[WeightProj] = weight_gradient(flat(operand), grad, proj_type);
        }
        if (!one_input) result[Residual] = grads[1];
        if (!input) return result;
        const at::Tensor back = (has_proj ? weight_proj : weight).unpack(self).t();
        at::Tensor skip = one_input ? grads[1] : at::Tensor();
        const auto whole = [&](const at::Tensor &t) { return t.view({kept.length, kept.batch, back.size(1)}); };
        if (!skip.defined()) {
            result[Input] = whole(at::mm(grad, back)).to(input_type);
        } else if (at::GradMode::is_enabled()) {
            result[Input] = skip + whole(at::mm(grad, back)).to(input_type);
        } else if (skip.scalar_type() == grad.scalar_type()) {
            skip.view({rows, back.size(1)}).addmm_(grad, back);
            result[Input] = skip;
        } else {
            result[Input] = skip.add_(whole(at::mm(grad, back)));
        }
        return result;
    }
};

// layer(input, residual, weight_proj, weight, weight_c, bias, init, act, d, bidirectional, has_skip, scale, mask_c, mask_pad)
//   -> (h, last) in the graph, or None: not the plain case, or no gradients are recorded
PyObject *layer(PyObject *, PyObject *const *a, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    Call c;
    Arg input, weight_proj, weight;
    if (observed() || !at::GradMode::is_enabled() || n != 14 || !read(a[0], input) || !read(a[1], c.x) || !read(a[2], weight_proj) || !read(a[3], weight) ||
        !read(a[4], c.weight_c) || !read(a[5], c.bias) || !read(a[6], c.init) || !read(a[7], c.act) || !read(a[8], c.d) || !read(a[9], c.bidirectional) ||
        !read(a[10], c.has_skip) || !read(a[11], c.scale) || !read(a[12], c.mask_c) || !read(a[13], c.pad) || !input || !weight || !c.weight_c ||
        !c.bias || !c.x || c.x->dim() != 3 || input->dim() != 3 || !input->is_cuda() || input->size(0) != c.x->size(0) || input->size(1) != c.x->size(1))
        return none();
    if (!(wants(input) || wants(c.x) || wants(weight_proj) || wants(weight) || wants(c.weight_c) || wants(c.bias) || wants(c.init))) return none();
    const bool autocast = at::autocast::is_autocast_enabled(at::kCUDA);
    const at::ScalarType type = autocast ? at::autocast::get_autocast_dtype(at::kCUDA) : input->scalar_type();
    int32_t code = 0;
    if (!dtype_code(type, code) || (autocast && !narrow(type))) return none();
    const c10::Device device = input->device();
    c.length = input->size(0);
    c.batch = input->size(1);
    const int64_t rows = c.length * c.batch, in = input->size(2);
    if (rows < 1 || in < 1 || !input->is_contiguous() || !aligned(*input.t, 16) || input->is_conj() || input->is_neg()) return none();
    int64_t inner = in;
    for (const Arg *w : {&weight_proj, &weight}) {
        if (!*w) continue;
        if ((*w)->dim() != 2 || (*w)->size(0) != inner || !plain(*w->t, device, (*w)->numel(), 16)) return none();
        inner = (*w)->size(1);
    }
    for (const Arg *t : {&input, &weight_proj, &weight})
        if (*t && (*t)->scalar_type() != type && !(autocast && (*t)->scalar_type() == at::kFloat)) return none();
    if (autocast && narrow(c.x->scalar_type()) && c.x->scalar_type() != type) return none();
    const Call given = c;
    at::Tensor operand = *input.t, proj_operand = variable(weight_proj), weight_operand = *weight.t, projected, u, h, last, states;
    int rc;
    {
        const Unlocked unlocked;
        const c10::DeviceGuard guard(device);
        u = at::empty({c.length, c.batch, inner}, input->options().dtype(type).requires_grad(false));
        c.u.t = &u;
        if (prepare(c, true, false)) {
            if (autocast) {   // (with gradients recorded: these are torch's own conversions, a parameter's made once in a region)
                operand = at::autocast::cached_cast(type, operand, at::kCUDA);
                if (weight_proj) proj_operand = at::autocast::cached_cast(type, proj_operand, at::kCUDA);
                weight_operand = at::autocast::cached_cast(type, weight_operand, at::kCUDA);
            }
            const at::AutoDispatchBelowADInplaceOrView below;
            const c10::impl::ExcludeDispatchKeyGuard as_they_are(c10::autocast_dispatch_keyset);
            at::Tensor x = operand.view({rows, in}), result = u.view({rows, inner});
            if (weight_proj) {
                projected = at::empty({rows, weight_proj->size(1)}, u.options());
                product_into(projected, x, proj_operand, code);
                x = projected;
            }
            product_into(result, x, weight_operand, code);
            rc = run_forward(c, true, h, last, states);
        } else {
            rc = -1;
        }
    }
    if (rc != SRU_AMD_OK) return none();
    const auto node = new_node<LayerNode>();
    const bool one_input = given.x.t->is_same(*input.t);
    node->set_next_edges(torch::autograd::collect_next_edges(*input.t, one_input || !c.x ? Variable() : *given.x.t, variable(weight_proj), *weight.t,
                                                             *given.weight_c.t, *given.bias.t, variable(given.init)));
    node->kept.keep(c, states);
    node->one_input = one_input;
    node->has_proj = (bool)weight_proj;
    node->input_type = input->scalar_type();
    node->weight_type = weight->scalar_type();
    if (weight_proj) node->proj_type = weight_proj->scalar_type();
    // (of the products' operands those that some gradient needs)
    const bool first = wants(input) || wants(weight_proj);
    if (weight_proj || wants(weight)) node->operand = SavedVariable(operand, false);
    if (weight_proj && wants(weight)) node->projected = SavedVariable(projected, false);
    if (weight_proj ? first : wants(input)) node->weight = SavedVariable(weight_operand, false);
    if (weight_proj) node->weight_proj = SavedVariable(proj_operand, false);
    torch::autograd::create_gradient_edge(h, node);
    torch::autograd::create_gradient_edge(last, node);
    return Py_BuildValue("(NN)", wrap(h), wrap(last));
    END_HANDLE_TH_ERRORS
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

// Whether what is launched now goes into a graph.
bool recorded(const c10::Device &device) {
    hipStreamCaptureStatus status = hipStreamCaptureStatusNone;
    if (hipStreamIsCapturing(c10::hip::getCurrentHIPStream(device.index()).stream(), &status) == hipSuccess) return status != hipStreamCaptureStatusNone;
    (void)hipGetLastError();   // (another stream is, and this is the one that all wait for)
    return false;
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
// in its form, or there is no kernel for the stack (or, in a graph, a slower one) or no room for its workspace
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
    // Another thread may give a cell another parameter, or a parameter other memory, while this one is unlocked.
    c10::Storage held[kLayers][5];
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
            if (need == 0 || (!sru_amd_stack_wanted_in_graph(&s, layers, n_proj) && recorded(device))) return none();
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
        c10::Storage *hold = held[l];
        for (const Arg *t : {&proj, &weight, &weight_c, &bias, &scale})
            if (*t) *hold++ = (*t)->storage();
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
        try {
            h = at::empty({length, batch, width}, options);
            last = at::empty({layers, batch, width}, options);
            const at::Tensor workspace = at::empty({(int64_t)need / 4}, options.dtype(at::kFloat));
            rc = sru_amd_stack_forward(&s, flags | SRU_AMD_SMALL_LAST, layers, n_proj, x.ptr(), projs, weights, wcs, biases, scales, init.ptr(),
                                       static_cast<const uint8_t *>(pad.ptr()), h.data_ptr(), last.data_ptr(), workspace.data_ptr(), need, stream_of(device));
        } catch (const c10::OutOfMemoryError &) {   // (layer by layer there is less at a time)
            rc = SRU_AMD_ERR_WORKSPACE;
        }
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
    {"recurrence", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(recurrence)), METH_FASTCALL, nullptr},
    {"layer", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(layer)), METH_FASTCALL, nullptr},
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
