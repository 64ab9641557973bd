// The per-call host path of heron_amd/hostops.py on torch tensors, as a CPython extension: operand checks, result allocation,
// problem description and launch in one native call.  The same steps in Python and ctypes cost 7 - 8 us a call beside the
// 2.5 us of the launch itself, more than most kernels of small products run.
//
// Every function takes the plain case only - contiguous device tensors of the instance's types and fitting shapes - and
// returns None for anything else, which hostops.py then handles (and words the error); a launch that the library refuses
// returns its error code.
#include <Python.h>

#include <algorithm>
#include <initializer_list>

#include <ATen/ATen.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include "../../include/heron_rocm.h"

namespace {

// integer argument i (None and wrong types leave a Python error set)
bool ints(PyObject* const* args, int from, int count, int64_t* out) {
    for (int i = 0; i < count; ++i) {
        out[i] = PyLong_AsLongLong(args[from + i]);
        if (out[i] == -1 && PyErr_Occurred()) return false;
    }
    return true;
}

// an int or a (height, width) pair
bool pair(PyObject* o, int64_t* h, int64_t* w) {
    if (PyTuple_Check(o) && PyTuple_GET_SIZE(o) == 2) {
        *h = PyLong_AsLongLong(PyTuple_GET_ITEM(o, 0));
        *w = PyLong_AsLongLong(PyTuple_GET_ITEM(o, 1));
    } else {
        *h = *w = PyLong_AsLongLong(o);
    }
    return !PyErr_Occurred();
}

const at::Tensor* tensor(PyObject* o) { return THPVariable_Check(o) ? &THPVariable_Unpack(o) : nullptr; }

bool is(const at::Tensor* t, at::ScalarType dt) { return t && t->is_cuda() && t->scalar_type() == dt && t->is_contiguous(); }

// a caller's result tensor: None, or on the operands' device, of the result's type, contiguous and large enough
bool result_fits(PyObject* o, const at::Tensor& operand, at::ScalarType dt, std::initializer_list<int64_t> shape) {
    if (o == Py_None) return true;
    const at::Tensor* t = tensor(o);
    if (!is(t, dt) || t->device() != operand.device()) return false;
    int64_t room = t->numel();
    for (int64_t d : shape) room /= d;                          // (the product of the extents may not fit)
    return room >= 1;
}

bool fits_int(int64_t v) { return v > 0 && v <= INT32_MAX; }

void* stream() { return (void*)c10::hip::getCurrentHIPStream().stream(); }

// A loaded instance: the handle and the descriptor (addresses, the tuple that Module hands over).
struct Instance {
    const hrn_module* mod;
    const hrn_kernel_desc* desc;
    at::ScalarType a, b, c;
    bool read(PyObject* native) {
        if (!PyTuple_Check(native) || PyTuple_GET_SIZE(native) != 2) return false;
        mod = (const hrn_module*)PyLong_AsVoidPtr(PyTuple_GET_ITEM(native, 0));
        desc = (const hrn_kernel_desc*)PyLong_AsVoidPtr(PyTuple_GET_ITEM(native, 1));
        if (PyErr_Occurred() || !desc) return false;
        const bool f16 = desc->dtype == HRN_DT_F16;
        a = f16 ? at::kHalf : at::kByte;
        b = f16 ? at::kHalf : at::kChar;
        c = f16 ? at::kHalf : at::kInt;
        return true;
    }
};

// What a launch may need besides its operands, alive until the call returns (torch's allocator hands the memory on in
// stream order): split-K partial sums, column sums of B that the caller did not bring.
struct Extras {
    at::Tensor workspace, bsum;
    int add(const Instance& in, hrn_problem* p, const at::Tensor& B, const at::Tensor* sums, int64_t split_k) {
        p->split_k = (int32_t)split_k;
        if (in.desc->split_k) {
            if (p->split_k < 1) p->split_k = 1;
            const int64_t need = hrn_splitk_workspace_fast_bytes(in.desc, p);
            if (need < 0) return (int)need;
            workspace = at::empty({need}, B.options().dtype(at::kByte));
            p->workspace = workspace.data_ptr();
            p->workspace_bytes = (size_t)need;
        }
        if (in.desc->colsum) {
            if (sums) {
                p->bsum = sums->data_ptr();
            } else {
                bsum = at::empty({(int64_t)p->batch * p->n}, B.options().dtype(at::kInt));
                p->bsum = bsum.data_ptr();
                return hrn_colsum_s8(B.data_ptr(), bsum.data_ptr(), p->batch, p->n, p->k, p->ldb,
                                     p->op == HRN_OP_GEMM ? p->stride_b : 0, stream());
            }
        }
        return HRN_OK;
    }
};

// the column sums argument: None, or (colsum instances) int32 sums of every column
bool sums_fit(const Instance& in, PyObject* o, int64_t columns) {
    if (o == Py_None || !in.desc->colsum) return true;
    const at::Tensor* t = tensor(o);
    return is(t, at::kInt) && t->numel() == columns;
}

// The interpreter lock, given up while the native part of a call runs: allocation and launch can wait for the driver or for
// room in a hardware queue, and other Python threads go on meanwhile.  Also taken back when an exception passes.  The caller
// holds the arguments, so their tensors stay.
struct Unlocked {
    PyThreadState* state = PyEval_SaveThread();
    ~Unlocked() { PyEval_RestoreThread(state); }
};

// C++ exceptions become the Python ones that torch makes of them (torch.OutOfMemoryError when the allocator is out of memory).
template <class F>
PyObject* guarded(F f) {
    try {
        return f();
    } catch (...) {
        torch::translate_exception_to_python(std::current_exception());
        return nullptr;
    }
}

// gemm(native, group_m, split_k, A, B, out, bsum)
PyObject* gemm(PyObject*, PyObject* const* args, Py_ssize_t n) {
    return guarded([&]() -> PyObject* {
        Instance in;
        int64_t v[2];
        if (n != 7 || !in.read(args[0]) || !ints(args, 1, 2, v)) {
            PyErr_Clear();
            Py_RETURN_NONE;
        }
        const at::Tensor *A = tensor(args[3]), *B = tensor(args[4]);
        if (!is(A, in.a) || !is(B, in.b) || A->dim() != B->dim() || (A->dim() != 2 && A->dim() != 3)) Py_RETURN_NONE;
        const int d = (int)A->dim() - 2;
        const int64_t batch = d ? A->size(0) : 1, M = A->size(d), K = A->size(d + 1), N = B->size(d);
        if (B->size(d + 1) != K || (d && B->size(0) != batch) || !fits_int(batch) || !fits_int(M) || !fits_int(N) || !fits_int(K) ||
            !sums_fit(in, args[6], batch * N))
            Py_RETURN_NONE;
        if (!result_fits(args[5], *A, in.c, {batch, M, N})) Py_RETURN_NONE;
        const at::Tensor* sums = tensor(args[6]);
        at::Tensor C;
        if (args[5] != Py_None) C = *tensor(args[5]);
        int rc;
        {
            Unlocked unlocked;
            if (!C.defined()) C = d ? at::empty({batch, M, N}, A->options().dtype(in.c)) : at::empty({M, N}, A->options().dtype(in.c));
            hrn_problem p;
            hrn_problem_gemm(&p, (int)batch, (int)M, (int)N, (int)K);
            p.group_m = (int32_t)v[0];
            Extras x;
            rc = x.add(in, &p, *B, sums, v[1]);
            if (rc == HRN_OK)
                rc = in.desc->dtype == HRN_DT_F16 ? hrn_launch_bmm_f16(in.mod, &p, A->data_ptr(), B->data_ptr(), C.data_ptr(), stream())
                                                  : hrn_launch_bmm_u8s8(in.mod, &p, A->data_ptr(), B->data_ptr(), C.data_ptr(), stream());
        }
        return rc == HRN_OK ? THPVariable_Wrap(C) : PyLong_FromLong(rc);
    });
}

// conv2d(native, group_m, split_k, X, W, stride, pad, dil, out, bsum)
PyObject* conv2d(PyObject*, PyObject* const* args, Py_ssize_t n) {
    return guarded([&]() -> PyObject* {
        Instance in;
        int64_t v[2], sh, sw, ph, pw, dh, dw;
        if (n != 10 || !in.read(args[0]) || !ints(args, 1, 2, v) || !pair(args[5], &sh, &sw) || !pair(args[6], &ph, &pw) ||
            !pair(args[7], &dh, &dw)) {
            PyErr_Clear();
            Py_RETURN_NONE;
        }
        const at::Tensor *X = tensor(args[3]), *W = tensor(args[4]);
        if (!is(X, in.a) || !is(W, in.b) || X->dim() != 4 || W->dim() != 4 || X->size(3) != W->size(3) || sh < 1 || sw < 1 || ph < 0 ||
            pw < 0 || dh < 1 || dw < 1 || !sums_fit(in, args[9], W->size(0)))
            Py_RETURN_NONE;
        for (int i = 0; i < 4; ++i)
            if (!fits_int(X->size(i)) || !fits_int(W->size(i))) Py_RETURN_NONE;
        if (std::max({sh, sw, ph, pw, dh, dw}) > 1 << 20) Py_RETURN_NONE;
        const int64_t room_h = X->size(1) - ((W->size(1) - 1) * dh + 1) + 2 * ph, room_w = X->size(2) - ((W->size(2) - 1) * dw + 1) + 2 * pw;
        if (room_h < 0 || room_w < 0) Py_RETURN_NONE;           // (before the division, which truncates)
        const int64_t ho = room_h / sh + 1, wo = room_w / sw + 1;
        if (!result_fits(args[8], *X, in.c, {X->size(0), ho, wo, W->size(0)})) Py_RETURN_NONE;
        const at::Tensor* sums = tensor(args[9]);
        at::Tensor C;
        if (args[8] != Py_None) C = *tensor(args[8]);
        int rc;
        {
            Unlocked unlocked;
            if (!C.defined()) C = at::empty({X->size(0), ho, wo, W->size(0)}, X->options().dtype(in.c));
            hrn_problem p;
            hrn_problem_conv2d_hw(&p, (int)X->size(0), (int)X->size(1), (int)X->size(2), (int)X->size(3), (int)W->size(0),
                                  (int)W->size(1), (int)W->size(2), (int)sh, (int)sw, (int)ph, (int)pw, (int)dh, (int)dw);
            p.group_m = (int32_t)v[0];
            Extras x;
            rc = x.add(in, &p, *W, sums, v[1]);
            if (rc == HRN_OK)
                rc = in.desc->dtype == HRN_DT_F16 ? hrn_launch_conv2d_nhwc_f16(in.mod, &p, X->data_ptr(), W->data_ptr(), C.data_ptr(), stream())
                                                  : hrn_launch_conv2d_nhwc_u8s8(in.mod, &p, X->data_ptr(), W->data_ptr(), C.data_ptr(), stream());
        }
        return rc == HRN_OK ? THPVariable_Wrap(C) : PyLong_FromLong(rc);
    });
}

// stream(): the current stream's handle
PyObject* current_stream(PyObject*, PyObject*) {
    return guarded([&]() -> PyObject* { return PyLong_FromVoidPtr(stream()); });
}

PyMethodDef methods[] = {
    {"gemm", (PyCFunction)(void (*)(void))gemm, METH_FASTCALL, "gemm(native, group_m, split_k, A, B, out, bsum)"},
    {"conv2d", (PyCFunction)(void (*)(void))conv2d, METH_FASTCALL, "conv2d(native, group_m, split_k, X, W, stride, pad, dil, out, bsum)"},
    {"stream", current_stream, METH_NOARGS, "handle of torch's current stream"},
    {nullptr, nullptr, 0, nullptr}};

PyModuleDef module_def = {PyModuleDef_HEAD_INIT, "_hrn_torch", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__hrn_torch(void) { return PyModule_Create(&module_def); }
