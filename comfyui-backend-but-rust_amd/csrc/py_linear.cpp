// qlinear.linear_w8a8's call as native code: the checks, the output's allocation and the launch of gpu_linear_w8a8 behind one call from
// Python.  3 x 256 -> 18432 takes 4.1 us on the GPU with weights that it has just read and 4.7 with 20 of them in turn (replayed from a
// graph); checked, allocated and called from Python it took 8.7 us of host time (a tensor 1.5, the call through ctypes with its 13 arguments
// about 2, attribute reads and checks the rest), this way 4.7.  A call in a row of them 8.1 and 4.9 us, bound by both sides alike.
//
// It answers None for whatever it does not take (a check that fails, tensor subclasses, modes and transforms that want to see the
// calls, return codes other than 0), and the caller then does the whole call in Python, which raises what there is to raise.
#include <ATen/core/Tensor.h>
#include <ATen/ops/empty.h>
#include <ATen/PythonTorchFunctionTLS.h>
#include <c10/core/impl/LocalDispatchKeySet.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Dtype.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include "../../include/gpu_api.h"

namespace {

int dt_of(at::ScalarType t) { return t == at::kFloat ? 0 : t == at::kHalf ? 1 : t == at::kBFloat16 ? 2 : -1; }

// Somebody wants to see tensor operations: their answers may be tensors without memory.
bool observed() {
    return c10::impl::TorchDispatchModeTLS::any_modes_set() || at::impl::torch_function_mode_enabled() ||
           c10::impl::tls_is_dispatch_key_included(c10::DispatchKey::FuncTorchDynamicLayerFrontMode) ||
           c10::impl::tls_is_dispatch_key_included(c10::DispatchKey::FuncTorchDynamicLayerBackMode);
}

const at::Tensor* plain(PyObject* o) { return THPVariable_CheckExact(o) ? &THPVariable_Unpack(o) : nullptr; }
bool dense(const at::Tensor& t, at::ScalarType type) { return t.is_cuda() && t.scalar_type() == type && t.is_contiguous(); }

// linear_w8a8(x, W, ws, bias, rotate, out_dtype) -> tensor, or None
PyObject* linear_w8a8(PyObject*, PyObject* const* args, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    if (n != 6 || !PyLong_CheckExact(args[4]) || observed()) Py_RETURN_NONE;
    const at::Tensor *x = plain(args[0]), *W = plain(args[1]), *ws = plain(args[2]), *bias = args[3] == Py_None ? nullptr : plain(args[3]);
    if (!x || !W || !ws || (args[3] != Py_None && !bias)) Py_RETURN_NONE;
    const at::ScalarType xt = x->scalar_type(), ot = args[5] == Py_None ? xt : THPDtype_Check(args[5]) ? ((THPDtype*)args[5])->scalar_type : at::kLong;
    if (!x->is_cuda() || x->layout() != at::kStrided || x->dim() != 2 || x->stride(1) != 1 || dt_of(xt) < 0 || dt_of(ot) < 0) Py_RETURN_NONE;
    if (!dense(*W, at::kChar) || !dense(*ws, at::kFloat) || (bias && !dense(*bias, ot)) || W->dim() != 2 || W->size(1) != x->size(1)) Py_RETURN_NONE;
    const int64_t M = x->size(0), K = x->size(1), N = W->size(0);
    int overflow = 0;
    const long rotate = PyLong_AsLongAndOverflow(args[4], &overflow);
    if (M < 1 || K < 1 || N < 1 || overflow || rotate != (int)rotate) Py_RETURN_NONE;
    at::Tensor D = at::empty({M, N}, x->options().dtype(ot).requires_grad(false)), scratch;
    const auto call = [&]() {
        const void *xp = x->data_ptr(), *bp = bias ? bias->data_ptr() : nullptr;
        void *dp = D.data_ptr(), *sp = scratch.defined() ? scratch.data_ptr() : nullptr;
        const int8_t* wp = (const int8_t*)W->data_ptr();
        const float* sc = (const float*)ws->data_ptr();
        if (!xp || !wp || !sc || !dp) return -1;
        void* stream = (void*)c10::hip::getCurrentHIPStream().stream();
        const int64_t stride = x->stride(0);
        int rc;
        Py_BEGIN_ALLOW_THREADS
        rc = gpu_linear_w8a8(dt_of(xt), xp, stride, wp, sc, bp, dp, sp, M, N, K, (int)rotate, dt_of(ot), stream);
        Py_END_ALLOW_THREADS
        return rc;
    };
    // a few short rows run as one kernel, which takes no scratch: without one the call either does that or queues nothing
    if (M <= 8 && K <= 1024 && call() == 0) return THPVariable_Wrap(std::move(D));
    scratch = at::empty({M * K + 4 * M}, x->options().dtype(at::kByte).requires_grad(false));   // codes and row scales
    if (call() == 0) return THPVariable_Wrap(std::move(D));
    Py_RETURN_NONE;
    END_HANDLE_TH_ERRORS
}

PyMethodDef methods[] = {{"linear_w8a8", (PyCFunction)(void (*)(void))linear_w8a8, METH_FASTCALL, nullptr}, {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_pycalls", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__pycalls() { return PyModule_Create(&module); }
