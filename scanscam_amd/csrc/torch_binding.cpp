// The op's host path in native code: what hip.scan_forward / hip.scan_backward do for plain GPU tensors -- checks,
// layout, outputs, workspace, stream, launch -- in one call from Python. At [4, 256, 1024] fp32 those steps took 13.5 us
// forward and 16.8 us backward in Python, several times the scan itself (4.8 / 6.0 us), and take 4.6 and 5.4 us here,
// the launch included; a training step through the op 67 -> 38 us where the autograd engine's thread wakes at once,
// 141 -> 64 us where it does not and the two threads pass the interpreter lock back and forth.
//
// scan(gate, value) is the whole op, its autograd node included. The node saves gate and output as the Python one does (hooks
// on saved tensors, version checks and the release after a backward pass are the engine's own), and its backward pass takes
// no interpreter lock: the same step 72 -> 55 us where the engine's thread does not wake at once (two wake-ups are most of
// what is left), the forward pass alone 8.0 -> 5.9 us and without gradients 6.3 -> 3.8 us ([8, 256, 32]).
//
// scan(gate, value), forward(gate, value) and backward(gate, output, out_grad) return None for every call they do not cover,
// and the caller goes on with the Python path, which also raises the errors: tensor subclasses and modes, functorch and fake
// tensors, forward-mode gradients, tracing, mismatched arguments, empty tensors, and views that have to be copied first. The
// library's entry points are handed in as addresses by bind(), so that whichever build of it hip.py loaded is the one that
// runs.
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/custom_function.h>
#include <torch/csrc/autograd/python_cpp_function.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/jit/frontend/tracer.h>
#include <torch/csrc/utils/pybind.h>

#include <ATen/PythonTorchFunctionTLS.h>
#include <ATen/record_function.h>
#include <ATen/ops/empty.h>
#include <c10/core/DeviceGuard.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <c10/hip/HIPStream.h>

#include <array>
#include <atomic>
#include <unordered_map>

#include "scanscam_hip.h"

namespace {

decltype(&scanscam_scan_fwd_strided) fwd_rows = nullptr;
decltype(&scanscam_scan_bwd_strided) bwd_rows = nullptr;
decltype(&scanscam_scan_fwd_cl_strided) fwd_cl = nullptr;
decltype(&scanscam_scan_bwd_cl_strided) bwd_cl = nullptr;
decltype(&scanscam_workspace_bytes) ws_rows = nullptr;
decltype(&scanscam_workspace_bytes_cl) ws_cl = nullptr;
decltype(&scanscam_strerror) error_text = nullptr;

// What scan()'s backward pass calls for gradients that the native path does not cover (bind(); never released).
PyObject *python_backward = nullptr;
// Calls are left to the Python path while it checks waits or limits polls (hip.check_waits).
std::atomic<bool> left_to_python{false};

constexpr int kMaxDims = 16;

int dtype_code(at::ScalarType t)
{
    switch (t) {
    case at::kFloat: return SCANSCAM_F32;
    case at::kBFloat16: return SCANSCAM_BF16;
    case at::kHalf: return SCANSCAM_F16;
    case at::kDouble: return SCANSCAM_F64;
    default: return -1;
    }
}

// A strided GPU tensor with memory of its own and nothing on top of it that a plain pointer would bypass.
bool plain(const at::Tensor &t)
{
    using K = c10::DispatchKey;
    constexpr c10::DispatchKeySet wrapped({K::Python, K::PythonTLSSnapshot, K::FuncTorchBatched, K::FuncTorchGradWrapper,
                                           K::FuncTorchVmapMode, K::Functionalize, K::Negative, K::Conjugate, K::ZeroTensor});
    return t.defined() && t.is_cuda() && t.layout() == at::kStrided && !t.key_set().has_any(wrapped) && t.has_storage();
}

struct Call {
    std::array<at::Tensor, 5> t;  // forward: gate, value, out; backward: gate, output, out_grad, gate_grad, value_grad
    int inputs, outputs;
    int code;
    bool cl;                      // channels-last
    int64_t n0, n1, T, C;         // rows: n0 groups of n1 rows of T; channels-last: n0 batch elements of [T, C]
    bool dense;
    std::array<scanscam_strides, 5> st;

    bool row_view(const at::Tensor &x) const { return x.size(-1) == 1 || x.stride(-1) == 1; }
    bool cl_view(const at::Tensor &x) const { return x.size(-2) > 1 && x.stride(-2) == 1 && !row_view(x); }

    // Inputs that this path takes as they are.
    bool accept()
    {
        const at::Tensor &first = t[0];
        const int64_t dims = first.dim();
        code = dtype_code(first.scalar_type());
        if (code < 0 || dims < 2 || dims > kMaxDims || first.numel() == 0) return false;
        for (int i = 0; i < inputs; i++) {
            if (!plain(t[i])) return false;
            if (i > 0 && (t[i].device() != first.device() || t[i].scalar_type() != first.scalar_type() || t[i].sizes() != first.sizes()))
                return false;
        }
        T = first.size(-1);
        cl = cl_view(t[0]) && cl_view(t[1]);  // (the rule looks at gate and value, or gate and output)
        if (cl) {
            C = first.size(-2);
            for (int i = 2; i < inputs; i++)
                if (!cl_view(t[i])) return false;
        } else {
            for (int i = 0; i < inputs; i++)
                if (!row_view(t[i])) return false;
        }
        return true;
    }

    void allocate()
    {
        const at::Tensor &first = t[0];
        const auto options = at::TensorOptions().dtype(first.scalar_type()).device(first.device());
        std::array<int64_t, kMaxDims> sizes;
        const int64_t dims = first.dim();
        for (int64_t d = 0; d < dims; d++) sizes[d] = first.size(d);
        if (cl) std::swap(sizes[dims - 1], sizes[dims - 2]);
        for (int i = inputs; i < inputs + outputs; i++) {
            t[i] = at::empty(at::IntArrayRef(sizes.data(), dims), options);
            if (cl) t[i] = t[i].transpose(-1, -2);
        }
    }

    // The leading dimensions (all but the last `inner`) merged into as few levels as all tensors allow, into n0, n1 and
    // st; false if that takes more than `most` levels.
    bool merge(int inner, int most)
    {
        const int n = inputs + outputs;
        int64_t size[2] = {1, 1}, stride[2][5] = {};
        int levels = 0;
        for (int64_t d = 0; d < t[0].dim() - inner; d++) {
            const int64_t s = t[0].size(d);
            if (s == 1) continue;
            bool joins = levels > 0;
            for (int i = 0; i < n && joins; i++) joins = stride[levels - 1][i] == t[i].stride(d) * s;
            if (joins) {
                size[levels - 1] *= s;
            } else {
                if (levels == most) return false;
                size[levels++] = s;
            }
            for (int i = 0; i < n; i++) stride[levels - 1][i] = t[i].stride(d);
        }
        const int last = levels > 0 ? levels - 1 : 0;
        n0 = levels == 2 || inner == 2 ? size[0] : 1;
        n1 = inner == 2 ? 1 : size[last];
        for (int i = 0; i < n; i++) {
            if (inner == 2) st[i] = {stride[0][i], t[i].stride(-1)};
            else st[i] = {levels == 2 ? stride[0][i] : 0, stride[last][i]};
        }
        return true;
    }

    bool lay_out()
    {
        dense = false;
        if (cl) {
            const int64_t esize = (int64_t)t[0].element_size();
            for (int i = 0; i < inputs + outputs; i++)  // (further apart than the kernels address: copied first)
                if (t[i].stride(-1) >= (int64_t(1) << 31) / esize / 18 || C >= (int64_t(1) << 31) / esize) return false;
            return merge(2, 1);
        }
        dense = true;
        for (int i = 0; i < inputs; i++) dense = dense && t[i].is_contiguous();
        if (dense) {
            n0 = 1;
            n1 = t[0].numel() / T;
            return true;
        }
        return merge(1, 2);
    }

    size_t workspace_bytes() const
    {
        const int direction = inputs == 2 ? SCANSCAM_FORWARD : SCANSCAM_BACKWARD;
        if (!cl) return ws_rows(n0 * n1, T, code, direction);
        // The channels-last choice goes through a cost model: remembered, a pure function of the shape.
        struct Key {
            int64_t b, T, C;
            int what;
            bool operator==(const Key &o) const { return b == o.b && T == o.T && C == o.C && what == o.what; }
        };
        struct Hash {
            size_t operator()(const Key &k) const
            {
                return (size_t)((uint64_t)k.b * 0x9E3779B97F4A7C15ull ^ (uint64_t)k.T * 0xC2B2AE3D27D4EB4Full ^
                                (uint64_t)k.C * 0x165667B19E3779F9ull ^ (uint64_t)k.what);
            }
        };
        static thread_local std::unordered_map<Key, size_t, Hash> known;
        const Key key{n0, T, C, code * 2 + direction};
        const auto it = known.find(key);
        if (it != known.end()) return it->second;
        if (known.size() >= 4096) known.clear();
        const size_t n = ws_cl(n0, T, C, code, direction, nullptr);
        known.emplace(key, n);
        return n;
    }

    int launch()
    {
        const size_t bytes = workspace_bytes();
        at::Tensor ws;
        if (bytes != 0) ws = at::empty({(int64_t)bytes}, at::TensorOptions().dtype(at::kByte).device(t[0].device()));
        void *w = bytes != 0 ? ws.data_ptr() : nullptr;
        void *stream = c10::hip::getCurrentHIPStream(t[0].device().index()).stream();
        void *p[5];
        for (int i = 0; i < inputs + outputs; i++) p[i] = t[i].data_ptr();
        auto s = [&](int i) { return dense ? nullptr : &st[i]; };
        if (inputs == 2)
            return cl ? fwd_cl(p[0], p[1], p[2], s(0), s(1), s(2), n0, T, C, code, w, bytes, stream, nullptr)
                      : fwd_rows(p[0], p[1], p[2], s(0), s(1), s(2), n0, n1, T, code, w, bytes, stream, nullptr);
        return cl ? bwd_cl(p[0], p[1], p[2], p[3], p[4], s(0), s(1), s(2), s(3), s(4), n0, T, C, code, w, bytes, stream, nullptr)
                  : bwd_rows(p[0], p[1], p[2], p[3], p[4], s(0), s(1), s(2), s(3), s(4), n0, n1, T, code, w, bytes, stream, nullptr);
    }
};

// A Python-level function or dispatch mode sees the calls of the Python path; leave them to it.
bool modes_active()
{
    return at::impl::PythonTorchFunctionTLS::stack_len() > 0 || c10::impl::TorchDispatchModeTLS::any_modes_set();
}

// Runs an accepted call; false if it is not covered after all. The library's errors are exceptions.
bool perform(Call &c)
{
    const c10::DeviceGuard guard(c.t[0].device());
    c.allocate();
    if (!c.lay_out()) return false;
    const int rc = c.launch();
    if (rc != SCANSCAM_OK)
        throw std::runtime_error(std::string("scanscam_scan_") + (c.inputs == 2 ? "fwd" : "bwd") + (c.cl ? "_cl" : "") + "_strided: " + error_text(rc));
    return true;
}

// The same for a call of which only the inputs are there, in c.t.
bool execute(Call &c) { return c.accept() && perform(c); }

PyObject *run(PyObject *const *args, Py_ssize_t nargs, int inputs, int outputs)
{
    HANDLE_TH_ERRORS
    if (nargs != inputs || !fwd_rows || modes_active()) Py_RETURN_NONE;
    Call c;
    c.inputs = inputs;
    c.outputs = outputs;
    for (int i = 0; i < inputs; i++) {
        if (!THPVariable_CheckExact(args[i])) Py_RETURN_NONE;
        c.t[i] = THPVariable_Unpack(args[i]);
    }
    bool covered;
    {
        pybind11::gil_scoped_release no_gil;
        covered = execute(c);
    }
    if (!covered) Py_RETURN_NONE;
    if (outputs == 1) return THPVariable_Wrap(std::move(c.t[2]));
    pybind11::object ga = pybind11::reinterpret_steal<pybind11::object>(THPVariable_Wrap(std::move(c.t[3])));
    pybind11::object gb = pybind11::reinterpret_steal<pybind11::object>(THPVariable_Wrap(std::move(c.t[4])));
    return PyTuple_Pack(2, ga.ptr(), gb.ptr());
    END_HANDLE_TH_ERRORS
}

using torch::autograd::variable_list;

variable_list backward_in_python(const at::Tensor &gate, const at::Tensor &output, const at::Tensor &out_grad)
{
    pybind11::gil_scoped_acquire gil;
    variable_list grads(2);
    pybind11::object args[3], result;
    const at::Tensor *t[3] = {&gate, &output, &out_grad};
    for (int i = 0; i < 3; i++) args[i] = pybind11::reinterpret_steal<pybind11::object>(THPVariable_Wrap(*t[i]));
    result = pybind11::reinterpret_steal<pybind11::object>(
        PyObject_CallFunctionObjArgs(python_backward, args[0].ptr(), args[1].ptr(), args[2].ptr(), nullptr));
    if (!result) {
        python_error error;
        error.persist();
        throw error;
    }
    for (int i = 0; i < 2; i++) grads[i] = THPVariable_Unpack(PyTuple_GET_ITEM(result.ptr(), i));
    return grads;
}

struct ScanBackward : torch::autograd::Function<ScanBackward> {
    // `done`: the call, executed.
    static at::Tensor forward(torch::autograd::AutogradContext *ctx, const at::Tensor &gate, const at::Tensor &, Call *done)
    {
        ctx->save_for_backward({gate, done->t[2]});
        return done->t[2];
    }
    static variable_list backward(torch::autograd::AutogradContext *ctx, variable_list out_grads)
    {
        RECORD_FUNCTION("ScanBackward", c10::ArrayRef<const c10::IValue>{});
        const variable_list saved = ctx->get_saved_variables();
        variable_list grads;
        Call c;
        c.inputs = 3;
        c.outputs = 2;
        c.t[0] = saved[0];
        c.t[1] = saved[1];
        c.t[2] = out_grads[0];
        if (!left_to_python && !modes_active() && execute(c)) grads = {c.t[3], c.t[4]};
        else grads = backward_in_python(saved[0], saved[1], out_grads[0]);
        grads.emplace_back();  // none for `done`
        return grads;
    }
};

// What Python sees of the node (output.grad_fn): the name and the attributes that a Python function's node has, on top of a
// C++ node's.
using ScanNode = torch::autograd::CppNode<ScanBackward>;

ScanNode *scan_node(PyObject *self) { return static_cast<ScanNode *>(reinterpret_cast<torch::autograd::THPCppFunction *>(self)->cdata.get()); }

PyObject *node_name(PyObject *, PyObject *) { return PyUnicode_FromString("ScanBackward"); }

PyObject *node_saved_tensors(PyObject *self, void *)
{
    HANDLE_TH_ERRORS
    const variable_list saved = scan_node(self)->ctx_.get_saved_variables();
    pybind11::tuple out(saved.size());
    for (size_t i = 0; i < saved.size(); i++) out[i] = pybind11::reinterpret_steal<pybind11::object>(THPVariable_Wrap(saved[i]));
    return out.release().ptr();
    END_HANDLE_TH_ERRORS
}

PyObject *node_needs_input_grad(PyObject *self, void *)
{
    ScanNode *node = scan_node(self);
    return PyTuple_Pack(2, node->should_compute_output(0) ? Py_True : Py_False, node->should_compute_output(1) ? Py_True : Py_False);
}

PyMethodDef node_methods[] = {{"name", node_name, METH_NOARGS, nullptr}, {nullptr, nullptr, 0, nullptr}};
PyGetSetDef node_properties[] = {{"saved_tensors", node_saved_tensors, nullptr, nullptr, nullptr},
                                 {"needs_input_grad", node_needs_input_grad, nullptr, nullptr, nullptr},
                                 {nullptr, nullptr, nullptr, nullptr, nullptr}};
PyTypeObject node_type;

PyObject *scan(PyObject *, PyObject *const *args, Py_ssize_t nargs)
{
    HANDLE_TH_ERRORS
    if (nargs != 2 || !fwd_rows || left_to_python || modes_active() || torch::jit::tracer::isTracing() ||
        c10::impl::tls_is_dispatch_key_included(c10::DispatchKey::FuncTorchDynamicLayerFrontMode))
        Py_RETURN_NONE;
    Call c;
    c.inputs = 2;
    c.outputs = 1;
    for (int i = 0; i < 2; i++) {
        if (!THPVariable_CheckExact(args[i])) Py_RETURN_NONE;
        c.t[i] = THPVariable_Unpack(args[i]);
        if (c.t[i]._fw_grad(/*level=*/0).defined()) Py_RETURN_NONE;
    }
    if (!c.accept()) Py_RETURN_NONE;
    bool covered;
    {
        pybind11::gil_scoped_release no_gil;
        RECORD_FUNCTION("Scan", c10::ArrayRef<const c10::IValue>{});
        {
            const at::AutoGradMode no_grad(false);
            covered = perform(c);
        }
        if (covered && at::GradMode::is_enabled() && (c.t[0].requires_grad() || c.t[1].requires_grad()))
            c.t[2] = ScanBackward::apply(c.t[0], c.t[1], &c);
    }
    if (!covered) Py_RETURN_NONE;
    return THPVariable_Wrap(std::move(c.t[2]));
    END_HANDLE_TH_ERRORS
}

PyObject *leave_to_python(PyObject *, PyObject *on)
{
    left_to_python = PyObject_IsTrue(on) == 1;
    Py_RETURN_NONE;
}

PyObject *forward(PyObject *, PyObject *const *args, Py_ssize_t nargs) { return run(args, nargs, 2, 1); }
PyObject *backward(PyObject *, PyObject *const *args, Py_ssize_t nargs) { return run(args, nargs, 3, 2); }

// bind(fwd_rows, bwd_rows, fwd_cl, bwd_cl, ws_rows, ws_cl, strerror, backward): addresses of the library's entry points, and
// the Python function (gate, output, out_grad) -> (gate_grad, value_grad). Returns the type of the autograd nodes.
PyObject *bind(PyObject *, PyObject *args)
{
    unsigned long long a[7];
    PyObject *callable;
    if (!PyArg_ParseTuple(args, "KKKKKKKO", a, a + 1, a + 2, a + 3, a + 4, a + 5, a + 6, &callable)) return nullptr;
    Py_INCREF(callable);
    python_backward = callable;
    bwd_rows = reinterpret_cast<decltype(bwd_rows)>(a[1]);
    fwd_cl = reinterpret_cast<decltype(fwd_cl)>(a[2]);
    bwd_cl = reinterpret_cast<decltype(bwd_cl)>(a[3]);
    ws_rows = reinterpret_cast<decltype(ws_rows)>(a[4]);
    ws_cl = reinterpret_cast<decltype(ws_cl)>(a[5]);
    error_text = reinterpret_cast<decltype(error_text)>(a[6]);
    fwd_rows = reinterpret_cast<decltype(fwd_rows)>(a[0]);
    static const bool registered = [] {
        // The type of a node whose class has none of its own.
        const std::shared_ptr<torch::autograd::Node> node(new ScanNode, torch::autograd::deleteNode);
        PyObject *plain_node = torch::autograd::functionToPyObject(node);
        node_type.tp_base = Py_TYPE(plain_node);
        Py_INCREF(node_type.tp_base);
        Py_DECREF(plain_node);
        torch::autograd::_initFunctionPyTypeObject(node_type, "ScanBackward", node_properties, node_methods);
        torch::autograd::registerCppFunction(typeid(ScanNode), &node_type);
        return true;
    }();
    (void)registered;
    Py_INCREF(&node_type);
    return reinterpret_cast<PyObject *>(&node_type);
}

PyMethodDef methods[] = {{"scan", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(scan)), METH_FASTCALL, nullptr},
                         {"leave_to_python", leave_to_python, METH_O, nullptr},
                         {"forward", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(forward)), METH_FASTCALL, nullptr},
                         {"backward", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(backward)), METH_FASTCALL, nullptr},
                         {"bind", bind, METH_VARARGS, nullptr},
                         {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_binding", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__binding()
{
    PyObject *m = PyModule_Create(&module);
    // The PyTorch it was compiled against, for hip.py to compare: its C++ API is not stable between versions.
    if (m && PyModule_AddStringConstant(m, "torch_version", SCANSCAM_TORCH_VERSION) != 0) Py_CLEAR(m);
    return m;
}
