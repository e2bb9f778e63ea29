// Host side of one QuantLinear call on the HIP backend, as a CPython module
// (qwen_int4_hip._host): the checks, the output and the call into the C ABI that
// qwen_int4_hip.backends.hip_w4g64_linear makes, without the interpreter.
//
// linear(x, qweight, scales, zeros, bias, out_features, in_features,
//        workspaces, grow) returns the output tensor, an int (the non-zero
// status of the C call) or None.  None means that the call is not of the plain
// form below; nothing has been done then, and the Python route takes it,
// raises what there is to raise and copies what there is to copy.
//
// Plain form: strided GPU tensors without subclass, mode, tracing or functorch
// level; contiguous, x and qweight 16-byte aligned, all on the current device;
// sizes and types of the canonical W4G64 contract; at least one row.
//
// What it measured: a call whose kernel takes 3 us cost 20.4 us of interpreter
// and ctypes time one after the other (1 x 1536 x 1536), now 7.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <ATen/PythonTorchFunctionTLS.h>
#include <ATen/core/Tensor.h>
#include <ATen/hip/impl/HIPStreamMasqueradingAsCUDA.h>
#include <ATen/ops/empty.h>
#include <c10/core/impl/LocalDispatchKeySet.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <c10/hip/HIPFunctions.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/jit/frontend/tracer.h>

#include "../../include/w4g64.h"

namespace {

int dtype_code(at::ScalarType t) {
    switch (t) {
        case at::kHalf: return W4G64_DTYPE_F16;
        case at::kBFloat16: return W4G64_DTYPE_BF16;
        case at::kFloat: return W4G64_DTYPE_F32;
        default: return W4G64_DTYPE_NONE;
    }
}

// The tensor behind `obj` if it is a plain GPU tensor (torch.Tensor itself or
// a Parameter, with storage of its own), else null.
const at::Tensor* plain(PyObject* obj) {
    if (!THPVariable_CheckExact(obj)) return nullptr;
    const at::Tensor& t = THPVariable_Unpack(obj);
    if (!t.defined() || !t.is_cuda() || t.layout() != at::kStrided || !t.has_storage() || t.is_conj() || t.is_neg() ||
        !t.is_contiguous() || t.unsafeGetTensorImpl()->is_python_dispatch())
        return nullptr;
    return &t;
}

bool plain_state() {
    return !at::impl::torch_function_mode_enabled() && c10::impl::TorchDispatchModeTLS::stack_len() == 0 &&
           !torch::jit::tracer::isTracing() &&
           !c10::impl::tls_is_dispatch_key_included(c10::DispatchKey::FuncTorchDynamicLayerFrontMode);
}

PyObject* linear(PyObject*, PyObject* const* args, Py_ssize_t count) {
    if (count != 9) {
        PyErr_SetString(PyExc_TypeError, "linear takes 9 arguments");
        return nullptr;
    }
    try {
        if (!PyLong_CheckExact(args[5]) || !PyLong_CheckExact(args[6]) || !plain_state()) Py_RETURN_NONE;
        const int64_t n = PyLong_AsLongLong(args[5]), k = PyLong_AsLongLong(args[6]);
        if (PyErr_Occurred()) {
            PyErr_Clear();
            Py_RETURN_NONE;
        }
        const at::Tensor *x = plain(args[0]), *qweight = plain(args[1]), *scales = plain(args[2]), *zeros = plain(args[3]);
        const at::Tensor* bias = args[4] == Py_None ? nullptr : plain(args[4]);
        if (!x || !qweight || !scales || !zeros || (args[4] != Py_None && !bias)) Py_RETURN_NONE;
        if (n <= 0 || k <= 0 || k % 64 || n > (int64_t(1) << 30) || k > (int64_t(1) << 30)) Py_RETURN_NONE;
        const int64_t groups = k / 64;
        const int x_code = dtype_code(x->scalar_type());
        const int bias_code = bias ? dtype_code(bias->scalar_type()) : W4G64_DTYPE_NONE;
        if (x_code == W4G64_DTYPE_NONE || x->dim() < 1 || x->size(-1) != k || x->numel() == 0 ||
            qweight->scalar_type() != at::kByte || qweight->numel() != n * k / 2 ||
            scales->scalar_type() != at::kHalf || scales->dim() != 2 || scales->size(0) != n ||
            scales->size(1) != groups || zeros->scalar_type() != at::kByte ||
            zeros->numel() != (n * groups + 1) / 2 ||
            (bias && (bias_code == W4G64_DTYPE_NONE || bias->dim() != 1 || bias->size(0) != n)))
            Py_RETURN_NONE;
        const c10::Device device = x->device();
        if (qweight->device() != device || scales->device() != device || zeros->device() != device ||
            (bias && bias->device() != device) || c10::hip::current_device() != device.index())
            Py_RETURN_NONE;
        const void* xp = x->const_data_ptr();
        const void* qp = qweight->const_data_ptr();
        if (((uintptr_t)xp | (uintptr_t)qp) & 15) Py_RETURN_NONE;

        const int64_t rows = x->numel() / k;
        hipStream_t stream = c10::hip::getCurrentHIPStreamMasqueradingAsCUDA(device.index()).stream();
        const int64_t need = w4g64_linear_workspace_bytes(rows, n, k, x_code);
        // The workspace of (device, stream), as kernels._workspace keeps it
        // (looked up under the GIL; `grow` makes or replaces it).
        void* workspace = nullptr;
        int64_t workspace_bytes = 0;
        PyObject* held = nullptr;  // the buffer, kept alive over the call
        if (need > 0) {
            PyObject* key = Py_BuildValue("(iK)", (int)device.index(), (unsigned long long)(uintptr_t)stream);
            if (!key) return nullptr;
            held = PyDict_GetItemWithError(args[7], key);
            Py_DECREF(key);
            if (!held && PyErr_Occurred()) return nullptr;
            if (held && THPVariable_Check(held) && THPVariable_Unpack(held).numel() >= need) {
                Py_INCREF(held);
            } else {
                held = PyObject_CallFunction(args[8], "L", (long long)need);
                if (!held) return nullptr;
                if (!THPVariable_Check(held)) {
                    Py_DECREF(held);
                    Py_RETURN_NONE;
                }
            }
            const at::Tensor& buffer = THPVariable_Unpack(held);
            workspace = buffer.data_ptr();
            workspace_bytes = buffer.numel();
        }
        int status = 0;
        at::Tensor y;
        try {
            auto sizes = x->sizes().vec();
            sizes.back() = n;
            y = at::empty(sizes, x->options().requires_grad(false));
            PyThreadState* save = PyEval_SaveThread();
            status = w4g64_linear(xp, x_code, (const uint8_t*)qp, (const uint16_t*)scales->const_data_ptr(),
                                  (const uint8_t*)zeros->const_data_ptr(), bias ? bias->const_data_ptr() : nullptr,
                                  bias_code, y.mutable_data_ptr(), rows, n, k, workspace, workspace_bytes, stream);
            PyEval_RestoreThread(save);
        } catch (...) {
            Py_XDECREF(held);
            throw;
        }
        Py_XDECREF(held);
        if (status) return PyLong_FromLong(status);
        return THPVariable_Wrap(y);
    } catch (...) {  // as torch's own bindings raise it (an allocation that failed)
        if (!PyErr_Occurred()) torch::translate_exception_to_python(std::current_exception());
        return nullptr;
    }
}

PyMethodDef kMethods[] = {
    {"linear", (PyCFunction)(void (*)(void))linear, METH_FASTCALL, "One W4G64 linear call; None: not of the plain form."},
    {nullptr, nullptr, 0, nullptr}};
PyModuleDef kModule = {PyModuleDef_HEAD_INIT, "_host", nullptr, -1, kMethods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__host(void) { return PyModule_Create(&kModule); }
