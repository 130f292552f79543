// The autograd operators on libgridnet_hip.so, natively: what backend_cuda.py and layernorm.py do
// per call from Python (argument checks, allocations, one ctypes call of sixteen arguments, the
// same again from autograd's thread with the interpreter lock) in C++.  On a small grid that host
// work is the call: 32^3, batch 2, ten inner iterations, forward + backward with a queue that
// never empties took 175 us for 79 us of kernels through Python.
//
// The functions here take only calls that are in order.  Anything else (a shape, dtype or device
// that does not fit, an empty batch, host tensors, an unknown activation) makes them return None:
// the Python operator is then called with the same arguments and raises, or handles it.  So does whatever
// torch does to an autograd.Function and these functions would go round: forward-mode derivatives,
// function transforms, tracing, dispatch modes, tensor subclasses (see tensor_arg and only_eager).
//
// The gradient buffers are handed to the library uninitialised with its overwrite flags; the Python
// operators' zero fills (four kernels per backward) have nothing to add to.
//
// Plain CPython functions with positional arguments (METH_FASTCALL) and autograd nodes of their own:
// pybind11's argument casters and torch::autograd::Function's boxed state cost more than the rest.

#include <c10/core/DeviceGuard.h>
#include <c10/core/impl/LocalDispatchKeySet.h>
#include <c10/hip/HIPStream.h>
#include <dlfcn.h>
#include <torch/csrc/autograd/functions/utils.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/autograd/saved_variable.h>
#include <torch/csrc/Exceptions.h>
#include <torch/torch.h>

#include <stdexcept>
#include <string>
#include <unordered_map>

#include "../../include/gridnet_hip.h"

namespace {

using at::Tensor;
using torch::autograd::Node;
using torch::autograd::SavedVariable;
using torch::autograd::variable_list;

// The library is bound by path and not by linking: the same file that the ctypes binding loaded
// (the caller may have pointed it at another build), and so the same error buffer.
struct Library {
    decltype(&gridnet_hip_version) version;
    decltype(&gridnet_hip_last_error) last_error;
    decltype(&gridnet_hip_forward) forward;
    decltype(&gridnet_hip_backward_workspace_bytes) backward_workspace_bytes;
    decltype(&gridnet_hip_backward) backward;
    decltype(&gridnet_hip_forward_gated) forward_gated;
    decltype(&gridnet_hip_backward_gated_workspace_bytes) backward_gated_workspace_bytes;
    decltype(&gridnet_hip_backward_gated) backward_gated;
    decltype(&gridnet_hip_layernorm_workspace_bytes) layernorm_workspace_bytes;
    decltype(&gridnet_hip_layernorm_forward) layernorm_forward;
    decltype(&gridnet_hip_layernorm_backward) layernorm_backward;
} lib;

void check(int status) {
    if (status != 0) throw std::runtime_error(lib.last_error());
}

int dtype_of(const Tensor &t) {
    switch (t.scalar_type()) {
        case at::kFloat: return GRIDNET_F32;
        case at::kDouble: return GRIDNET_F64;
        default: return -1;
    }
}

int activation_of(PyObject *name) {
    if (!PyUnicode_Check(name)) return -1;
    if (!PyUnicode_CompareWithASCIIString(name, "silu")) return GRIDNET_ACT_SILU;
    if (!PyUnicode_CompareWithASCIIString(name, "leaky_relu")) return GRIDNET_ACT_LEAKY_RELU;
    if (!PyUnicode_CompareWithASCIIString(name, "relu")) return GRIDNET_ACT_RELU;
    if (!PyUnicode_CompareWithASCIIString(name, "tanh")) return GRIDNET_ACT_TANH;
    return -1;
}

void *stream_of(const Tensor &t) { return c10::hip::getCurrentHIPStream(t.device().index()).stream(); }

Tensor workspace(size_t bytes, const Tensor &like) {
    return at::empty({(int64_t)(bytes ? bytes : 1)}, like.options().dtype(at::kByte).requires_grad(false));
}

Tensor fresh(const Tensor &like) { return at::empty(like.sizes(), like.options().requires_grad(false)); }

// contiguous, of x's dtype, on x's device
bool goes_with(const Tensor &t, const Tensor &x) {
    return t.defined() && t.is_contiguous() && t.scalar_type() == x.scalar_type() && t.device() == x.device();
}

bool usable_input(const Tensor &x) {
    return x.defined() && x.is_cuda() && x.is_contiguous() && x.dim() == 4 && x.numel() > 0 && dtype_of(x) >= 0;
}

// sizes of t: `lead...`, then the last three of x
bool shaped(const Tensor &t, std::initializer_list<int64_t> lead, const Tensor &x) {
    const auto s = t.sizes(), g = x.sizes();
    if (s.size() != lead.size() + 3) return false;
    size_t i = 0;
    for (int64_t n : lead)
        if (s[i++] != n) return false;
    return s[i] == g[1] && s[i + 1] == g[2] && s[i + 2] == g[3];
}

bool wants_graph(std::initializer_list<const Tensor *> inputs) {
    if (!at::GradMode::is_enabled()) return false;
    for (const Tensor *t : inputs)
        if (t->requires_grad()) return true;
    return false;
}

// The gradient that came in, as the kernels take it; the Python operators' checks and message.
const Tensor &incoming(const Tensor &g, const Tensor &like) {
    if (!g.is_cuda()) throw std::runtime_error("outGrads must be a CUDA tensor");
    if (!g.is_contiguous()) throw std::runtime_error("outGrads must be contiguous");
    if (g.scalar_type() != like.scalar_type() || g.device() != like.device() || g.sizes() != like.sizes())
        throw std::runtime_error("outGrads does not match the output in shape, dtype or device");
    return g;
}

struct StepShape {
    int dt, B, M, N, K, inner, bs, normalize, act;
    double eps;
};

struct StepNode : public Node {
    SavedVariable weight, bias, scale, x;
    StepShape p;
    std::string name() const override { return "GridnetStepBackward"; }
    void release_variables() override {
        weight.reset_data();
        bias.reset_data();
        scale.reset_data();
        x.reset_data();
    }
    variable_list apply(variable_list &&grads) override {
        if (!grads[0].defined()) return variable_list(4);
        const Tensor w = weight.unpack(), b = bias.unpack(), r = scale.unpack(), xs = x.unpack();
        c10::DeviceGuard guard(xs.device());
        const Tensor &g = incoming(grads[0], xs);
        Tensor dw = fresh(w), db = fresh(b), dr = fresh(b), dx = fresh(xs);
        const size_t bytes = lib.backward_workspace_bytes(p.dt, p.B, p.M, p.N, p.K, p.inner, p.bs, p.normalize);
        const Tensor ws = workspace(bytes, xs);
        check(lib.backward(p.dt, w.data_ptr(), b.data_ptr(), r.data_ptr(), xs.data_ptr(), g.data_ptr(), dw.data_ptr(),
                           db.data_ptr(), dr.data_ptr(), dx.data_ptr(), p.B, p.M, p.N, p.K, p.inner, p.bs, p.eps,
                           p.normalize, p.act, GRIDNET_OVERWRITE, ws.data_ptr(), bytes, stream_of(xs)));
        return {dw, db, dr, dx};
    }
};

struct GatedNode : public Node {
    SavedVariable weight, bias, x;
    StepShape p;
    std::string name() const override { return "GatedGridnetStepBackward"; }
    void release_variables() override {
        weight.reset_data();
        bias.reset_data();
        x.reset_data();
    }
    variable_list apply(variable_list &&grads) override {
        if (!grads[0].defined()) return variable_list(3);
        const Tensor w = weight.unpack(), b = bias.unpack(), xs = x.unpack();
        c10::DeviceGuard guard(xs.device());
        const Tensor &g = incoming(grads[0], xs);
        Tensor dw = fresh(w), db = fresh(b), dx = fresh(xs);
        const size_t bytes = lib.backward_gated_workspace_bytes(p.dt, p.B, p.M, p.N, p.K, p.inner, p.bs);
        const Tensor ws = workspace(bytes, xs);
        check(lib.backward_gated(p.dt, w.data_ptr(), b.data_ptr(), xs.data_ptr(), g.data_ptr(), dw.data_ptr(),
                                 db.data_ptr(), dx.data_ptr(), p.B, p.M, p.N, p.K, p.inner, p.bs, p.act,
                                 GRIDNET_OVERWRITE, ws.data_ptr(), bytes, stream_of(xs)));
        return {dw, db, dx};
    }
};

struct NormNode : public Node {
    SavedVariable x, gamma, mean, rstd;
    std::string name() const override { return "GridLayerNormBackward"; }
    void release_variables() override {
        x.reset_data();
        gamma.reset_data();
        mean.reset_data();
        rstd.reset_data();
    }
    variable_list apply(variable_list &&grads) override {
        if (!grads[0].defined()) return variable_list(3);
        const Tensor xs = x.unpack(), ga = gamma.unpack(), m = mean.unpack(), r = rstd.unpack();
        c10::DeviceGuard guard(xs.device());
        const Tensor g = grads[0].contiguous();
        Tensor dx = fresh(xs), dgamma = fresh(ga), dbeta = fresh(ga);
        const int dt = dtype_of(xs), B = (int)xs.size(0);
        const long n = ga.numel();
        const size_t bytes = lib.layernorm_workspace_bytes(dt, B, n);
        const Tensor ws = workspace(bytes, xs);
        check(lib.layernorm_backward(dt, g.data_ptr(), xs.data_ptr(), ga.data_ptr(), m.data_ptr(), r.data_ptr(),
                                     dx.data_ptr(), dgamma.data_ptr(), dbeta.data_ptr(), B, n, GRIDNET_OVERWRITE_PARAMS,
                                     ws.data_ptr(), bytes, stream_of(xs)));
        return {dx, dgamma, dbeta};
    }
};

template <typename N> std::shared_ptr<N> make_node() {
    return std::shared_ptr<N>(new N(), torch::autograd::deleteNode);
}

// The interpreter lock is given up while kernels are launched: a full queue makes a launch wait.
struct WithoutGil {
    PyThreadState *state = PyEval_SaveThread();
    ~WithoutGil() { PyEval_RestoreThread(state); }
};

// Nothing but eager execution and autograd would see this call: no dispatch mode, functorch transform or
// tracer on this thread.
bool only_eager() {
    constexpr c10::DispatchKeySet usual({c10::DispatchKey::BackendSelect, c10::DispatchKey::ADInplaceOrView});
    return (c10::impl::tls_local_dispatch_key_set().included_ - usual).empty();
}

// An ordinary device tensor (or Parameter): no subclass, no wrapper of a transform, no lazy negation, and no
// tangent of forward-mode differentiation, which these operators have no rule for.
const Tensor *tensor_arg(PyObject *o) {
    constexpr c10::DispatchKeySet usual({c10::DispatchKey::CUDA, c10::DispatchKey::AutogradCUDA,
                                         c10::DispatchKey::AutocastCUDA, c10::DispatchKey::ADInplaceOrView});
    if (!THPVariable_CheckExact(o)) return nullptr;
    const Tensor &t = THPVariable_Unpack(o);
    if (!t.defined() || (t.key_set().raw_repr() & ~usual.raw_repr()) || t._fw_grad(0).defined()) return nullptr;
    return &t;
}

// Another number of arguments is no call to decline but another build than the Python files'.
constexpr char kArguments[] = "%s takes %d arguments, got %zd (a stale _torch_ops.so?)";

// (weight, bias, residual_scale, init_activations, inner, block_size, eps, normalize, activation)
PyObject *step(PyObject *, PyObject *const *args, Py_ssize_t nargs) {
    HANDLE_TH_ERRORS
    if (nargs != 9) return PyErr_Format(PyExc_TypeError, kArguments, "step", 9, nargs);
    if (!only_eager()) Py_RETURN_NONE;
    const Tensor *w = tensor_arg(args[0]), *b = tensor_arg(args[1]), *r = tensor_arg(args[2]), *x = tensor_arg(args[3]);
    if (!w || !b || !r || !x || !usable_input(*x) || !goes_with(*w, *x) || !goes_with(*b, *x) || !goes_with(*r, *x) ||
        !shaped(*w, {27}, *x) || !shaped(*b, {}, *x) || !shaped(*r, {}, *x))
        Py_RETURN_NONE;
    StepShape p{};
    p.inner = (int)PyLong_AsLong(args[4]);
    p.bs = (int)PyLong_AsLong(args[5]);
    p.eps = PyFloat_AsDouble(args[6]);
    p.normalize = PyObject_IsTrue(args[7]);
    p.act = activation_of(args[8]);
    if (PyErr_Occurred()) {
        PyErr_Clear();
        Py_RETURN_NONE;
    }
    const auto s = x->sizes();
    p.dt = dtype_of(*x);
    p.B = (int)s[0]; p.M = (int)s[1]; p.N = (int)s[2]; p.K = (int)s[3];
    if (p.act < 0 || p.bs <= 0 || p.M % p.bs || p.N % p.bs || p.K % p.bs) Py_RETURN_NONE;
    c10::DeviceGuard guard(x->device());
    Tensor y = fresh(*x);
    int status;
    {
        WithoutGil unlocked;
        status = lib.forward(p.dt, w->data_ptr(), b->data_ptr(), r->data_ptr(), x->data_ptr(), y.data_ptr(), p.B, p.M, p.N, p.K,
                      p.inner, p.bs, p.eps, p.normalize, p.act, stream_of(*x));
    }
    check(status);
    if (wants_graph({w, b, r, x})) {
        auto node = make_node<StepNode>();
        node->set_next_edges(torch::autograd::collect_next_edges(*w, *b, *r, *x));
        node->weight = SavedVariable(*w, false);
        node->bias = SavedVariable(*b, false);
        node->scale = SavedVariable(*r, false);
        node->x = SavedVariable(*x, false);
        node->p = p;
        torch::autograd::set_history(y, node);
    }
    return THPVariable_Wrap(std::move(y));
    END_HANDLE_TH_ERRORS
}

// (weight, bias, init_activations, inner, block_size, activation)
PyObject *gated_step(PyObject *, PyObject *const *args, Py_ssize_t nargs) {
    HANDLE_TH_ERRORS
    if (nargs != 6) return PyErr_Format(PyExc_TypeError, kArguments, "gated_step", 6, nargs);
    if (!only_eager()) Py_RETURN_NONE;
    const Tensor *w = tensor_arg(args[0]), *b = tensor_arg(args[1]), *x = tensor_arg(args[2]);
    if (!w || !b || !x || !usable_input(*x) || !goes_with(*w, *x) || !goes_with(*b, *x) || !shaped(*w, {27, 2}, *x) ||
        !shaped(*b, {2}, *x))
        Py_RETURN_NONE;
    StepShape p{};
    p.inner = (int)PyLong_AsLong(args[3]);
    p.bs = (int)PyLong_AsLong(args[4]);
    p.act = activation_of(args[5]);
    if (PyErr_Occurred()) {
        PyErr_Clear();
        Py_RETURN_NONE;
    }
    const auto s = x->sizes();
    p.dt = dtype_of(*x);
    p.B = (int)s[0]; p.M = (int)s[1]; p.N = (int)s[2]; p.K = (int)s[3];
    if (p.act < 0 || p.bs <= 0 || p.M % p.bs || p.N % p.bs || p.K % p.bs) Py_RETURN_NONE;
    c10::DeviceGuard guard(x->device());
    Tensor y = fresh(*x);
    int status;
    {
        WithoutGil unlocked;
        status = lib.forward_gated(p.dt, w->data_ptr(), b->data_ptr(), x->data_ptr(), y.data_ptr(), p.B, p.M, p.N, p.K, p.inner,
                            p.bs, p.act, stream_of(*x));
    }
    check(status);
    if (wants_graph({w, b, x})) {
        auto node = make_node<GatedNode>();
        node->set_next_edges(torch::autograd::collect_next_edges(*w, *b, *x));
        node->weight = SavedVariable(*w, false);
        node->bias = SavedVariable(*b, false);
        node->x = SavedVariable(*x, false);
        node->p = p;
        torch::autograd::set_history(y, node);
    }
    return THPVariable_Wrap(std::move(y));
    END_HANDLE_TH_ERRORS
}

// (x, weight, bias, eps)
PyObject *layer_norm(PyObject *, PyObject *const *args, Py_ssize_t nargs) {
    HANDLE_TH_ERRORS
    if (nargs != 4) return PyErr_Format(PyExc_TypeError, kArguments, "layer_norm", 4, nargs);
    if (!only_eager()) Py_RETURN_NONE;
    const Tensor *x = tensor_arg(args[0]), *ga = tensor_arg(args[1]), *be = tensor_arg(args[2]);
    if (!x || !ga || !be || !usable_input(*x) || !goes_with(*ga, *x) || !goes_with(*be, *x) || !shaped(*ga, {}, *x) ||
        !shaped(*be, {}, *x))
        Py_RETURN_NONE;
    const double eps = PyFloat_AsDouble(args[3]);
    if (PyErr_Occurred()) {
        PyErr_Clear();
        Py_RETURN_NONE;
    }
    c10::DeviceGuard guard(x->device());
    const int dt = dtype_of(*x), B = (int)x->size(0);
    const long n = ga->numel();
    Tensor y = fresh(*x);
    const auto opts = x->options().requires_grad(false);
    Tensor mean = at::empty({B}, opts), rstd = at::empty({B}, opts);
    const size_t bytes = lib.layernorm_workspace_bytes(dt, B, n);
    const Tensor ws = workspace(bytes, *x);
    int status;
    {
        WithoutGil unlocked;
        status = lib.layernorm_forward(dt, x->data_ptr(), ga->data_ptr(), be->data_ptr(), y.data_ptr(), mean.data_ptr(),
                                rstd.data_ptr(), B, n, eps, ws.data_ptr(), bytes, stream_of(*x));
    }
    check(status);
    if (wants_graph({x, ga, be})) {
        auto node = make_node<NormNode>();
        node->set_next_edges(torch::autograd::collect_next_edges(*x, *ga, *be));
        node->x = SavedVariable(*x, false);
        node->gamma = SavedVariable(*ga, false);
        node->mean = SavedVariable(mean, false);
        node->rstd = SavedVariable(rstd, false);
        torch::autograd::set_history(y, node);
    }
    return THPVariable_Wrap(std::move(y));
    END_HANDLE_TH_ERRORS
}

template <typename F> bool find(void *handle, const char *name, F &to) {
    to = reinterpret_cast<F>(dlsym(handle, name));
    if (!to) PyErr_Format(PyExc_ImportError, "the gridnet HIP library has no %s", name);
    return to != nullptr;
}

// Bind to the library at `path`.
PyObject *bind(PyObject *, PyObject *path) {
    const char *file = PyUnicode_AsUTF8(path);
    if (!file) return nullptr;
    void *h = dlopen(file, RTLD_NOW | RTLD_LOCAL);
    if (!h) return PyErr_Format(PyExc_ImportError, "cannot load %s: %s", file, dlerror());
#define GRIDNET_FIND(member) \
    if (!find(h, "gridnet_hip_" #member, lib.member)) return nullptr
    GRIDNET_FIND(version);
    if (lib.version() != GRIDNET_HIP_VERSION)  // built against another header than the library
        return PyErr_Format(PyExc_ImportError, "%s has version %d of the C ABI, _torch_ops.so was built for %d", file,
                            lib.version(), GRIDNET_HIP_VERSION);
    GRIDNET_FIND(last_error);
    GRIDNET_FIND(forward);
    GRIDNET_FIND(backward_workspace_bytes);
    GRIDNET_FIND(backward);
    GRIDNET_FIND(forward_gated);
    GRIDNET_FIND(backward_gated_workspace_bytes);
    GRIDNET_FIND(backward_gated);
    GRIDNET_FIND(layernorm_workspace_bytes);
    GRIDNET_FIND(layernorm_forward);
    GRIDNET_FIND(layernorm_backward);
#undef GRIDNET_FIND
    Py_RETURN_NONE;
}

PyMethodDef methods[] = {
    {"bind", bind, METH_O, nullptr},
    {"step", (PyCFunction)(void (*)(void))step, METH_FASTCALL, nullptr},
    {"gated_step", (PyCFunction)(void (*)(void))gated_step, METH_FASTCALL, nullptr},
    {"layer_norm", (PyCFunction)(void (*)(void))layer_norm, METH_FASTCALL, nullptr},
    {nullptr, nullptr, 0, nullptr},
};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_torch_ops", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__torch_ops() { return PyModule_Create(&module); }
