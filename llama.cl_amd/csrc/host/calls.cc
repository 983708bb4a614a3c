// fc_Q4A and attention_rope2 as the Python module calls them, in native code: the argument checks, the output and the
// call of the C entry.  A small call is shorter than the Python around it (one row of a 4096 x 4096 product: 5.4 us on the
// device, 10.9 us per call through ctypes and 5.2 us so; one token of attention over 2048 rows of halves 21.2 and 14.1).
//
// These are shortcuts for the ordinary case and decide nothing: whatever is not ordinary -- a tensor subclass, vmap, a mode
// that intercepts calls, a stream under capture, a workspace that is missing or too small, any argument that a check
// would refuse -- returns NotImplemented with nothing done, and the Python function takes the call, workspace policy and
// error messages included.  (torch.jit.trace does not stop them: neither way can it record more than the output's
// allocation.)  Nothing is kept between calls but the addresses of the C entries.
#include <Python.h>

#include <ATen/ATen.h>
#include <ATen/PythonTorchFunctionTLS.h>
#include <ATen/hip/HIPContext.h>
#include <c10/core/impl/LocalDispatchKeySet.h>
#include <c10/hip/HIPGraphsC10Utils.h>
#include <pybind11/pybind11.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include "../../../include/llmops_hip.h"

namespace {

decltype(&llmops_fc_Q4A_workspace_bytes) fc_workspace_bytes;
decltype(&llmops_fc_Q4A) fc;
decltype(&llmops_attention_workspace_bytes) attention_workspace_bytes;
decltype(&llmops_attention_rope) attention;
decltype(&llmops_last_error) last_error;

// a plain dense tensor with memory of its own on the HIP device
bool plain(PyObject* o, at::ScalarType type, int64_t dims) {
    if (!THPVariable_CheckExact(o)) return false;
    const at::Tensor& t = THPVariable_Unpack(o);
    using K = c10::DispatchKey;
    constexpr c10::DispatchKeySet kWrapped({K::Python, K::PythonTLSSnapshot, K::FuncTorchBatched, K::FuncTorchGradWrapper, K::Batched,
                                            K::Functionalize, K::Conjugate, K::Negative, K::ZeroTensor});
    return t.defined() && t.is_cuda() && t.layout() == at::kStrided && t.scalar_type() == type && t.dim() == dims &&
           !t.key_set().has_any(kWrapped) && t.has_storage() && t.is_contiguous();
}

// nothing between this call and the device: no Python mode, no functorch level, no capture on the stream
bool direct() {
    using K = c10::DispatchKey;
    constexpr c10::DispatchKeySet kModes({K::Python, K::PythonTLSSnapshot, K::FuncTorchDynamicLayerFrontMode, K::FuncTorchDynamicLayerBackMode,
                                          K::FuncTorchVmapMode, K::Batched, K::Functionalize});
    return !at::impl::torch_function_mode_enabled() && !c10::impl::tls_local_dispatch_key_set().included_.has_any(kModes) &&
           c10::hip::currentStreamCaptureStatusMayInitCtx() == c10::hip::CaptureStatus::None;
}

// the module's workspace of this family on this device and stream, undefined if there is none of `bytes`
at::Tensor workspace(PyObject* held, const char* kind, const at::Tensor& t, hipStream_t stream, size_t bytes) {
    PyObject* key = Py_BuildValue("(ssiK)", kind, "cuda", (int)t.get_device(), (unsigned long long)(uintptr_t)stream);
    if (key == nullptr) {
        PyErr_Clear();
        return {};
    }
    PyObject* ws = PyDict_Check(held) ? PyDict_GetItem(held, key) : nullptr;  // (borrowed)
    Py_DECREF(key);
    if (ws == nullptr || !THPVariable_CheckExact(ws)) return {};
    const at::Tensor& w = THPVariable_Unpack(ws);
    return (size_t)w.numel() >= bytes ? w : at::Tensor();
}

hipStream_t current_stream(const at::Tensor& t) { return c10::hip::getCurrentHIPStream(t.get_device()).stream(); }

PyObject* refused() {
    const char* what = last_error();
    PyErr_SetString(PyExc_RuntimeError, what);
    return nullptr;
}

PyObject* not_ordinary() { Py_RETURN_NOTIMPLEMENTED; }

// fc_Q4A(workspaces, input, weiq, N)
PyObject* call_fc(PyObject*, PyObject* const* args, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    if (n != 4 || !PyLong_CheckExact(args[3]) || !plain(args[1], at::kFloat, 3) || !plain(args[2], at::kChar, 3) || !direct())
        return not_ordinary();
    const at::Tensor &x = THPVariable_Unpack(args[1]), &w = THPVariable_Unpack(args[2]);
    int overflow = 0;
    const int64_t N = PyLong_AsLongLongAndOverflow(args[3], &overflow);
    const int64_t B = x.size(0), M = x.size(1), K = x.size(2), Ng = w.size(0), Kg = w.size(1), blk = w.size(2);
    const int g = blk == 640 ? 32 : blk == 2176 ? 128 : 0;
    if (overflow || g == 0 || N <= 0 || B <= 0 || M <= 0 || K <= 0) return not_ordinary();
    const hipStream_t st = current_stream(x);
    const at::Tensor ws = workspace(args[0], "fc", x, st, fc_workspace_bytes(B * M, K, Ng, Kg, g));
    if (!ws.defined()) return not_ordinary();
    at::Tensor y = at::empty({B, M, N}, x.options().requires_grad(false));
    int rc = 0;
    {
        pybind11::gil_scoped_release others_run;  // (a launch can wait for room in the queue)
        rc = fc(static_cast<const float*>(x.data_ptr()), B * M, K, static_cast<const int8_t*>(w.data_ptr()), Ng, Kg, g, N,
                static_cast<float*>(y.data_ptr()), ws.data_ptr(), (size_t)ws.numel(), st);
    }
    if (rc != 0) return refused();
    return THPVariable_Wrap(std::move(y));
    END_HANDLE_TH_ERRORS
}

// attention_rope2(workspaces, q, k, v, inv_freq, kv_cache, kvc_slots, position_id, layer_id)
PyObject* call_attention(PyObject*, PyObject* const* args, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    if (n != 9 || !plain(args[1], at::kFloat, 3) || !plain(args[2], at::kFloat, 3) || !plain(args[3], at::kFloat, 3) ||
        !plain(args[4], at::kFloat, 1) || !(plain(args[5], at::kFloat, 5) || plain(args[5], at::kHalf, 5)) || !plain(args[6], at::kInt, 1) ||
        !PyLong_CheckExact(args[7]) || !PyLong_CheckExact(args[8]) || !direct())
        return not_ordinary();
    const at::Tensor &q = THPVariable_Unpack(args[1]), &k = THPVariable_Unpack(args[2]), &v = THPVariable_Unpack(args[3]),
                     &f = THPVariable_Unpack(args[4]), &c = THPVariable_Unpack(args[5]), &slots = THPVariable_Unpack(args[6]);
    const int64_t B = q.size(0), qL = q.size(1), planes = c.size(0), H = c.size(2), maxlen = c.size(3), S = c.size(4);
    int over[2] = {0, 0};
    const long position = PyLong_AsLongAndOverflow(args[7], &over[0]), layer = PyLong_AsLongAndOverflow(args[8], &over[1]);
    if (over[0] || over[1] || position != (int)position || layer != (int)layer || c.size(1) != B || B <= 0 || qL <= 0 || q.size(2) != H * S ||
        k.sizes() != q.sizes() || v.sizes() != q.sizes() || slots.size(0) != qL)
        return not_ordinary();
    const hipStream_t st = current_stream(q);
    const at::Tensor ws = workspace(args[0], "attn", q, st, attention_workspace_bytes(B, qL, H, S, maxlen));
    if (!ws.defined()) return not_ordinary();
    int rc = 0;
    {
        pybind11::gil_scoped_release others_run;
        rc = attention(static_cast<float*>(q.data_ptr()), static_cast<float*>(k.data_ptr()), static_cast<const float*>(v.data_ptr()), B, qL, H, S,
                       static_cast<const float*>(f.data_ptr()), f.size(0), c.data_ptr(), c.scalar_type() == at::kFloat ? 0 : 1, planes, maxlen,
                       static_cast<const int32_t*>(slots.data_ptr()), (int)position, (int)layer, ws.data_ptr(), (size_t)ws.numel(), st);
    }
    if (rc != 0) return refused();
    Py_RETURN_NONE;
    END_HANDLE_TH_ERRORS
}

// bind(addresses of the C entries, in the order of the variables above)
PyObject* bind(PyObject*, PyObject* args) {
    unsigned long long a[5];
    if (!PyArg_ParseTuple(args, "KKKKK", &a[0], &a[1], &a[2], &a[3], &a[4])) return nullptr;
    fc_workspace_bytes = reinterpret_cast<decltype(fc_workspace_bytes)>((uintptr_t)a[0]);
    fc = reinterpret_cast<decltype(fc)>((uintptr_t)a[1]);
    attention_workspace_bytes = reinterpret_cast<decltype(attention_workspace_bytes)>((uintptr_t)a[2]);
    attention = reinterpret_cast<decltype(attention)>((uintptr_t)a[3]);
    last_error = reinterpret_cast<decltype(last_error)>((uintptr_t)a[4]);
    Py_RETURN_NONE;
}

PyMethodDef methods[] = {{"bind", bind, METH_VARARGS, nullptr},
                         {"fc_Q4A", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(call_fc)), METH_FASTCALL, nullptr},
                         {"attention_rope2", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(call_attention)), METH_FASTCALL, nullptr},
                         {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_host", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__host(void) {
    PyObject* m = PyModule_Create(&module);
    if (m != nullptr && PyModule_AddStringConstant(m, "built_for", LLMOPS_BUILT_FOR) != 0) {  // (compared before anything is called)
        Py_DECREF(m);
        return nullptr;
    }
    return m;
}
