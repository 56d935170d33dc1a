// The torch-facing wrappers of the small calls, in native code: argument checks, output tensors and the C ABI call of an operator that
// takes a few microseconds on the GPU cost several times that when every step of them is a Python call (4096 x 4096, one row: 31.7 us a
// pair of calls with ctypes and torch.zeros, two fill kernels among them). Each function returns its tensors, or the C ABI's error code
// as an int, which the Python side turns into its exception; what torch throws keeps its Python type (torch.OutOfMemoryError, IndexError, ...).
// Other Python threads run while a call allocates and enqueues.
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include <ATen/hip/impl/HIPStreamMasqueradingAsCUDA.h>
#include <ATen/ops/empty.h>

#include "mi355_strix.h"

namespace {

mi355_stream current_stream() { return c10::hip::getCurrentHIPStreamMasqueradingAsCUDA().stream(); }

// host: pinned host memory, which the GPU reaches, will do
bool tensor_arg(PyObject* o, const char* what, const at::Tensor*& t, bool host) {
    if (!THPVariable_Check(o)) { PyErr_Format(PyExc_TypeError, "%s must be a tensor", what); return false; }
    t = &THPVariable_Unpack(o);
    if (t->is_cuda() || (host && t->is_pinned())) return true;
    PyErr_Format(PyExc_RuntimeError, host ? "%s must be on the GPU or in pinned memory" : "%s must be on the GPU", what);
    return false;
}
bool unsigned_arg(PyObject* o, uint64_t& v) {
    v = PyLong_AsUnsignedLongLongMask(o);
    return !PyErr_Occurred();
}
bool truth_arg(PyObject* o, bool& v) {
    const int truth = PyObject_IsTrue(o);
    v = truth > 0;
    return truth >= 0;
}

// (x, want_sums) -> (codes, deltas, sums or None, status)
PyObject* quantize_a8(PyObject*, PyObject* const* args, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    const at::Tensor* x;
    if (n != 2) { PyErr_SetString(PyExc_TypeError, "quantize_a8 takes 2 arguments"); return nullptr; }
    if (!tensor_arg(args[0], "x", x, false)) return nullptr;
    if (x->dim() != 2 || x->stride(1) != 1) { PyErr_SetString(PyExc_AssertionError, "x must be rows of contiguous values"); return nullptr; }
    bool want_sums;
    if (!truth_arg(args[1], want_sums)) return nullptr;
    uint32_t kind;
    switch (x->scalar_type()) {
    case at::kFloat: kind = MI355_INPUT_F32; break;
    case at::kHalf: kind = MI355_INPUT_F16; break;
    case at::kBFloat16: kind = MI355_INPUT_BF16; break;
    default: PyErr_SetString(PyExc_KeyError, "x must be float32, float16 or bfloat16"); return nullptr;
    }
    at::Tensor codes, deltas, sums, status;
    int32_t rc;
    {
        pybind11::gil_scoped_release others;
        const int64_t rows = x->size(0), width = x->size(1), groups = width / 32;
        const auto like = x->options().requires_grad(false);
        codes = at::empty({rows, width}, like.dtype(at::kChar));
        deltas = at::empty({rows, groups}, like.dtype(at::kFloat));
        if (want_sums) sums = at::empty({rows, groups}, like.dtype(at::kInt));
        status = at::empty({rows}, like.dtype(at::kInt));
        if (width == 0) status.zero_();      // (no launch for rows without values)
        rc = mi355_quantize_a8_fresh(x->data_ptr(), kind, static_cast<uint32_t>(rows), static_cast<uint32_t>(width),
                                     static_cast<uint64_t>(x->stride(0)) * x->element_size(), static_cast<int8_t*>(codes.data_ptr()),
                                     static_cast<float*>(deltas.data_ptr()), want_sums ? static_cast<int32_t*>(sums.data_ptr()) : nullptr,
                                     static_cast<uint32_t*>(status.data_ptr()), current_stream());
    }
    if (rc != 0) return PyLong_FromLong(rc);
    PyObject* out = PyTuple_New(4);
    PyTuple_SET_ITEM(out, 0, THPVariable_Wrap(std::move(codes)));
    PyTuple_SET_ITEM(out, 1, THPVariable_Wrap(std::move(deltas)));
    if (want_sums) PyTuple_SET_ITEM(out, 2, THPVariable_Wrap(std::move(sums)));
    else { Py_INCREF(Py_None); PyTuple_SET_ITEM(out, 2, Py_None); }
    PyTuple_SET_ITEM(out, 3, THPVariable_Wrap(std::move(status)));
    return out;
    END_HANDLE_TH_ERRORS
}

// (weight, codes, deltas, n_in, count, out or None, accumulate, row_bytes, out_stride) -> out; row_bytes / out_stride 0: dense
PyObject* gemv_q8_0_a8(PyObject*, PyObject* const* args, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    const at::Tensor *weight, *codes, *deltas, *given = nullptr;
    uint64_t n_in, count, row_bytes, out_stride;
    bool accumulate;
    if (n != 9) { PyErr_SetString(PyExc_TypeError, "gemv_q8_0_a8 takes 9 arguments"); return nullptr; }
    // (an output made here lives where the codes do)
    if (!tensor_arg(args[0], "weight", weight, true) || !tensor_arg(args[1], "codes", codes, args[5] != Py_None) || !tensor_arg(args[2], "deltas", deltas, true) ||
        !unsigned_arg(args[3], n_in) || !unsigned_arg(args[4], count) || (args[5] != Py_None && !tensor_arg(args[5], "out", given, true)) ||
        !truth_arg(args[6], accumulate) || !unsigned_arg(args[7], row_bytes) || !unsigned_arg(args[8], out_stride))
        return nullptr;
    at::Tensor out;
    int32_t rc;
    {
        pybind11::gil_scoped_release others;
        const int64_t rows = codes->size(0);
        if (given) out = *given;
        else {
            out = at::empty({rows, static_cast<int64_t>(count)}, codes->options().requires_grad(false).dtype(at::kFloat));
            if (accumulate) out.zero_();     // (otherwise the launch writes every value)
        }
        const mi355_q8a8_view v{static_cast<const uint8_t*>(weight->data_ptr()), static_cast<const int8_t*>(codes->data_ptr()),
                                static_cast<const float*>(deltas->data_ptr()), static_cast<float*>(out.data_ptr()),
                                static_cast<uint32_t>(row_bytes ? row_bytes : n_in / 32U * 34U), static_cast<uint32_t>(n_in), static_cast<uint32_t>(count),
                                static_cast<uint32_t>(rows), static_cast<uint32_t>(codes->size(1)), static_cast<uint32_t>(out_stride ? out_stride : out.size(1)),
                                accumulate ? 1U : 0U};
        rc = mi355_gemv_q8_0_a8(&v, current_stream());
    }
    if (rc != 0) return PyLong_FromLong(rc);
    return THPVariable_Wrap(std::move(out));
    END_HANDLE_TH_ERRORS
}

PyMethodDef methods[] = {{"quantize_a8", reinterpret_cast<PyCFunction>(quantize_a8), METH_FASTCALL, nullptr},
                         {"gemv_q8_0_a8", reinterpret_cast<PyCFunction>(gemv_q8_0_a8), METH_FASTCALL, nullptr},
                         {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_torch_ops", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__torch_ops(void) { return PyModule_Create(&module); }
