// The operators of ops.py that serve decode batches, as one native call each: argument checks, the output and the workspace
// as torch tensors, the current stream and the library call.  The kernels of a linear of one token take 3.3 to 4.8 us; the same
// steps from Python took the host 9.5 us, most of it in three foreign-function calls with some twenty converted arguments: four linears
// of one token 40.1 us a pass that way, 22.2 us this way, of which the kernels are 16.
//
// A call takes what the operators are given in ordinary use and returns None for everything else - other layouts, tensor subclasses,
// modes that watch torch calls, tracing, wrapped tensors, a bias that torch follows -, which ops.py then does step by step, with
// the same result or the same error.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <ATen/PythonTorchFunctionTLS.h>
#include <ATen/core/Tensor.h>
#include <ATen/core/grad_mode.h>
#include <ATen/ops/empty.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Dtype.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/jit/frontend/tracer.h>
#include <torch/version.h>

#include "cosmos_fp8.h"

namespace {

// torch functions are watched or recorded: the step-by-step form lets the watcher see them
bool watched() {
    return at::impl::torch_function_mode_enabled() || c10::impl::TorchDispatchModeTLS::any_modes_set() || torch::jit::tracer::isTracing();
}

// torch.Tensor or Parameter itself, on the GPU, with memory of its own (not one of torch.func's wrappers)
bool plain(PyObject* obj, const at::Tensor*& t) {
    using c10::DispatchKey;
    static const c10::DispatchKeySet kWrapped({DispatchKey::FuncTorchBatched, DispatchKey::FuncTorchGradWrapper, DispatchKey::Batched, DispatchKey::Functionalize,
                                               DispatchKey::Python});
    if (!THPVariable_CheckExact(obj)) return false;
    t = &THPVariable_Unpack(obj);
    return t->defined() && !t->key_set().has_any(kWrapped) && t->is_cuda() && t->layout() == at::kStrided && t->has_storage() && !t->is_conj() && !t->is_neg();
}

bool out_code(PyObject* obj, at::ScalarType& type, int& code) {
    if (!THPDtype_Check(obj)) return false;
    type = reinterpret_cast<THPDtype*>(obj)->scalar_type;
    code = type == at::kBFloat16 ? CFP8_OUT_BF16 : CFP8_OUT_F32;
    return type == at::kBFloat16 || type == at::kFloat;
}

PyObject* failed(int rc) {
    const char* const msg = cfp8_last_error();
    if (rc == CFP8_EINVAL) PyErr_Format(PyExc_ValueError, "cosmos_fp8: %s", msg ? msg : "");
    else PyErr_Format(PyExc_RuntimeError, "cosmos_fp8 error %d: %s", rc, msg ? msg : "");
    return nullptr;
}

// fp8_linear(x, weight, weight_scale, bias, out_dtype)
PyObject* fp8_linear(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
    HANDLE_TH_ERRORS
    const at::Tensor *x, *w, *s, *b = nullptr;
    at::ScalarType type;
    int code;
    if (nargs != 5 || !plain(args[0], x) || !plain(args[1], w) || !plain(args[2], s) || !out_code(args[4], type, code) || watched()) Py_RETURN_NONE;
    if (x->dim() != 2 || w->dim() != 2 || x->scalar_type() != at::kBFloat16 || s->scalar_type() != at::kFloat || !s->is_contiguous()) Py_RETURN_NONE;
    const int64_t M = x->size(0), K = w->size(0), N = w->size(1);
    if (M < 1 || N < 1 || K < 2 || x->size(1) != K || x->stride(1) != 1 || w->stride(0) != 1) Py_RETURN_NONE;
    if (s->numel() < N || (w->scalar_type() != at::kFloat8_e4m3fn && w->scalar_type() != at::kByte)) Py_RETURN_NONE;
    if (args[3] != Py_None) {
        // what the GEMMs add themselves: one bf16 value a column that torch does not follow
        if (!plain(args[3], b) || b->scalar_type() != at::kBFloat16 || b->dim() != 1 || b->size(0) != N || b->stride(0) != 1 || b->device() != x->device()) Py_RETURN_NONE;
        if ((b->requires_grad() && at::GradMode::is_enabled()) || b->_fw_grad(0).defined() || (reinterpret_cast<uintptr_t>(b->data_ptr()) & 7u)) Py_RETURN_NONE;
    }
    at::Tensor out;
    int rc;
    {
        pybind11::gil_scoped_release no_gil;
        const size_t bytes = cfp8_linear_workspace_bytes(M, K) + cfp8_gemm_partial_bytes(CFP8_DISPATCH_ROWWISE, M, N, K);
        const at::Tensor work = at::empty({(int64_t)(bytes > 256 ? bytes : 256)}, x->options().dtype(at::kByte).requires_grad(false));
        out = at::empty({M, N}, x->options().dtype(type).requires_grad(false));
        rc = cfp8_linear_rowwise_split(x->data_ptr(), M > 1 ? x->stride(0) : K, w->data_ptr(), N > 1 ? w->stride(1) : K, s->data_ptr<float>(),
                                       b ? b->data_ptr() : nullptr, out.data_ptr(), N, code, M, N, K, work.data_ptr(), (size_t)work.numel(),
                                       c10::hip::getCurrentHIPStream().stream());
    }
    if (rc) return failed(rc);
    return THPVariable_Wrap(std::move(out));
    END_HANDLE_TH_ERRORS
}

// linear_mxfp4(x, codes, scales, out_dtype)
PyObject* linear_mxfp4(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
    HANDLE_TH_ERRORS
    const at::Tensor *x, *w, *s;
    at::ScalarType type;
    int code;
    if (nargs != 4 || !plain(args[0], x) || !plain(args[1], w) || !plain(args[2], s) || !out_code(args[3], type, code) || watched()) Py_RETURN_NONE;
    if (x->dim() != 2 || w->dim() != 2 || s->dim() != 2 || x->scalar_type() != at::kBFloat16 || w->scalar_type() != at::kByte || s->scalar_type() != at::kByte)
        Py_RETURN_NONE;
    const int64_t M = x->size(0), K = x->size(1), N = w->size(0);
    if (M < 1 || N < 1 || K < 32 || K % 32 || w->size(1) != K / 2 || s->size(0) != N || s->size(1) != K / 32 || !w->is_contiguous() || !s->is_contiguous()) Py_RETURN_NONE;
    if (x->stride(1) != 1 || x->stride(0) % 8 || (reinterpret_cast<uintptr_t>(x->data_ptr()) & 15u)) Py_RETURN_NONE;
    at::Tensor out;
    int rc;
    {
        pybind11::gil_scoped_release no_gil;
        // (up to 4 tokens on K up to 4096: one launch that takes no partial sums)
        const size_t bytes = cfp8_linear_workspace_bytes(M, K) + (M > 4 || K > 4096 ? cfp8_gemm_partial_bytes(CFP8_DISPATCH_MXFP4, M, N, K) : 0);
        const at::Tensor work = at::empty({(int64_t)(bytes > 1 ? bytes : 1)}, x->options().dtype(at::kByte).requires_grad(false));
        out = at::empty({M, N}, x->options().dtype(type).requires_grad(false));
        rc = cfp8_linear_mxfp4(x->data_ptr(), M > 1 ? x->stride(0) : K, w->data_ptr(), K / 2, s->data_ptr(), K / 32, out.data_ptr(), N, code, M, N, K,
                               work.data_ptr(), bytes, c10::hip::getCurrentHIPStream().stream());
    }
    if (rc) return failed(rc);
    return THPVariable_Wrap(std::move(out));
    END_HANDLE_TH_ERRORS
}

PyMethodDef kMethods[] = {
    {"fp8_linear", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(fp8_linear)), METH_FASTCALL, "x, weight, weight_scale, bias, out_dtype -> tensor or None"},
    {"linear_mxfp4", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(linear_mxfp4)), METH_FASTCALL, "x, codes, scales, out_dtype -> tensor or None"},
    {nullptr, nullptr, 0, nullptr}};

PyModuleDef kModule = {PyModuleDef_HEAD_INIT, "_torch_calls", nullptr, -1, kMethods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

#define CFP8_TEXT_OF(x) #x
#define CFP8_TEXT(x) CFP8_TEXT_OF(x)

PyMODINIT_FUNC PyInit__torch_calls() {
    PyObject* const module = PyModule_Create(&kModule);
    // (tensors are laid out as this torch has them: another one may load this file and read them wrongly)
    if (module && PyModule_AddStringConstant(module, "BUILT_FOR", "torch " TORCH_VERSION ", Python " CFP8_TEXT(PY_MAJOR_VERSION) "." CFP8_TEXT(PY_MINOR_VERSION)) < 0) {
        Py_DECREF(module);
        return nullptr;
    }
    return module;
}
