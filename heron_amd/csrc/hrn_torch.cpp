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

// ---- the passes and the channels-first launch of hostops.run_operator ----
// An eager conv3d spent 30 us of Python and ctypes on three kernels of 16 us.
bool plain(const at::Tensor* t) {
    return t && t->is_cuda() && t->is_contiguous() && (t->element_size() == 1 || t->element_size() == 2 || t->element_size() == 4);
}

// channels_last(x, cp): (N, C, L) -> (N, L, cp)
PyObject* channels_last(PyObject*, PyObject* const* args, Py_ssize_t n) {
    return guarded([&]() -> PyObject* {
        int64_t cp;
        if (n != 2 || !ints(args, 1, 1, &cp)) {
            PyErr_Clear();
            Py_RETURN_NONE;
        }
        const at::Tensor* x = tensor(args[0]);
        if (!plain(x) || x->dim() != 3) Py_RETURN_NONE;
        const int64_t N = x->size(0), C = x->size(1), L = x->size(2);
        if (!fits_int(N) || !fits_int(C) || !fits_int(L) || !fits_int(cp) || N > 65535) Py_RETURN_NONE;
        at::Tensor out;
        int rc;
        {
            Unlocked unlocked;
            out = at::empty({N, L, cp}, x->options());
            rc = hrn_transpose_pad(x->data_ptr(), out.data_ptr(), (int)N, (int)C, (int)L, (int)cp, (int)x->element_size(), stream());
        }
        return rc == HRN_OK ? THPVariable_Wrap(out) : PyLong_FromLong(rc);
    });
}

// integers of a tuple or list, at most `cap`; -1: something else
int int_list(PyObject* o, int64_t* out, int cap) {
    if (!PyTuple_Check(o) && !PyList_Check(o)) return -1;
    const Py_ssize_t n = PySequence_Fast_GET_SIZE(o);
    if (n > cap) return -1;
    for (Py_ssize_t i = 0; i < n; ++i) {
        out[i] = PyLong_AsLongLong(PySequence_Fast_GET_ITEM(o, i));
        if (out[i] == -1 && PyErr_Occurred()) return -1;
    }
    return (int)n;
}

// gather(src, out, dst_dim, coords, dst_stride, dst_live, op, aux): backend.make_gather and the pass; HRN_OK or its error code
PyObject* gather(PyObject*, PyObject* const* args, Py_ssize_t n) {
    return guarded([&]() -> PyObject* {
        hrn_gather g = {};
        int64_t op;
        auto parse = [&]() {
            if (n != 8 || !ints(args, 6, 1, &op)) return false;
            const int nd = int_list(args[2], g.dst_dim, HRN_GATHER_DIMS);
            if (nd < 1 || !PyList_Check(args[3])) return false;
            const Py_ssize_t ns = PyList_GET_SIZE(args[3]);
            if (ns < 1 || ns > HRN_GATHER_DIMS) return false;
            int64_t stride = 1;
            for (int d = nd - 1; d >= 0; --d) {
                g.dst_stride[d] = stride;
                g.dst_live[d] = g.dst_dim[d];
                stride *= g.dst_dim[d];
            }
            if (args[4] != Py_None && int_list(args[4], g.dst_stride, HRN_GATHER_DIMS) != nd) return false;
            if (args[5] != Py_None && int_list(args[5], g.dst_live, HRN_GATHER_DIMS) != nd) return false;
            for (Py_ssize_t s = 0; s < ns; ++s) {
                PyObject* e = PyList_GET_ITEM(args[3], s);
                if (!PyTuple_Check(e)) return false;
                const Py_ssize_t len = PyTuple_GET_SIZE(e);
                if (len < 3 || len > 5 || !PyDict_Check(PyTuple_GET_ITEM(e, 2))) return false;
                int64_t v[5] = {0, 0, 0, 0, 1};
                for (Py_ssize_t i = 0; i < len; ++i) {
                    if (i == 2) continue;
                    v[i] = PyLong_AsLongLong(PyTuple_GET_ITEM(e, i));
                    if (v[i] == -1 && PyErr_Occurred()) return false;
                }
                g.src_dim[s] = v[0]; g.src_stride[s] = v[1]; g.add[s] = v[3]; g.div[s] = v[4];
                PyObject *key, *val;
                Py_ssize_t pos = 0;
                while (PyDict_Next(PyTuple_GET_ITEM(e, 2), &pos, &key, &val)) {
                    const long long d = PyLong_AsLongLong(key), m = PyLong_AsLongLong(val);
                    if (PyErr_Occurred() || d < 0 || d >= nd) return false;
                    g.mul[s][d] = m;
                }
            }
            g.ndim = nd;
            g.nsrc = (int32_t)ns;
            g.op = (int32_t)op;
            return true;
        };
        const at::Tensor *src = n == 8 ? tensor(args[0]) : nullptr, *out = n == 8 ? tensor(args[1]) : nullptr;
        const at::Tensor* aux = n == 8 ? tensor(args[7]) : nullptr;
        if (!plain(src) || !plain(out) || (!aux && args[7] != Py_None) || (aux && !plain(aux)) || !parse()) {
            PyErr_Clear();
            Py_RETURN_NONE;
        }
        g.elem_bytes = (int32_t)src->element_size();
        int rc;
        {
            Unlocked unlocked;
            rc = hrn_gather_nd(&g, src->data_ptr(), aux ? aux->data_ptr() : nullptr, out->data_ptr(), stream());
        }
        return PyLong_FromLong(rc);
    });
}

// conv_chw(native, group_m, split_k, X, xshape, W, stride, pad, dil, view, shape, bsum): hrn_launch_conv2d_chw with a fresh result of
// `shape`; view: (expand, in_h, in_w, top, left)
PyObject* conv_chw(PyObject*, PyObject* const* args, Py_ssize_t n) {
    return guarded([&]() -> PyObject* {
        Instance in;
        int64_t v[2], x4[4], vw[5], shape[5], sh, sw, ph, pw, dh, dw;
        int dims = -1;
        if (n != 12 || !in.read(args[0]) || !ints(args, 1, 2, v) || int_list(args[4], x4, 4) != 4 || !pair(args[6], &sh, &sw) ||
            !pair(args[7], &ph, &pw) || !pair(args[8], &dh, &dw) || int_list(args[9], vw, 5) != 5 || (dims = int_list(args[10], shape, 5)) < 2) {
            PyErr_Clear();
            Py_RETURN_NONE;
        }
        const at::Tensor *X = tensor(args[3]), *W = tensor(args[5]);
        if (!is(X, in.a) || !is(W, in.b) || W->dim() != 4 || x4[3] != W->size(3) || sh < 1 || sw < 1 || ph < 0 || pw < 0 || dh < 1 || dw < 1 ||
            in.desc->split_k || !sums_fit(in, args[11], W->size(0)))
            Py_RETURN_NONE;
        for (int i = 0; i < 4; ++i)
            if (!fits_int(x4[i]) || !fits_int(W->size(i))) Py_RETURN_NONE;
        // (what is in memory: the pixels before the expansion)
        if (X->numel() != x4[0] * (vw[0] > 0 ? vw[1] * vw[2] : x4[1] * x4[2]) * x4[3]) Py_RETURN_NONE;
        if (std::max({sh, sw, ph, pw, dh, dw}) > 1 << 20) Py_RETURN_NONE;
        for (int64_t e : vw)
            if (e < 0 || e > INT32_MAX) Py_RETURN_NONE;
        hrn_problem p;
        hrn_problem_conv2d_hw(&p, (int)x4[0], (int)x4[1], (int)x4[2], (int)x4[3], (int)W->size(0), (int)W->size(1), (int)W->size(2), (int)sh,
                              (int)sw, (int)ph, (int)pw, (int)dh, (int)dw);
        p.group_m = (int32_t)v[0];
        int64_t count = 1;
        for (int i = 0; i < dims; ++i) {
            if (!fits_int(shape[i])) Py_RETURN_NONE;
            count *= shape[i];
            if (count > INT64_MAX >> 32) Py_RETURN_NONE;
        }
        if (p.m < 1 || count != (int64_t)p.m * p.n || p.m % shape[0]) Py_RETURN_NONE;
        hrn_conv_view view = {(int32_t)(p.m / shape[0]), (int32_t)vw[0], (int32_t)vw[1], (int32_t)vw[2], (int32_t)vw[3], (int32_t)vw[4]};
        const at::Tensor* sums = tensor(args[11]);
        at::Tensor C;
        int rc;
        {
            Unlocked unlocked;
            C = at::empty(at::IntArrayRef(shape, dims), X->options().dtype(in.c));
            Extras x;
            rc = x.add(in, &p, *W, sums, v[1]);
            if (rc == HRN_OK) rc = hrn_launch_conv2d_chw(in.mod, &p, &view, X->data_ptr(), W->data_ptr(), C.data_ptr(), stream());
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
    {"channels_last", (PyCFunction)(void (*)(void))channels_last, METH_FASTCALL, "channels_last(x, cp)"},
    {"gather", (PyCFunction)(void (*)(void))gather, METH_FASTCALL, "gather(src, out, dst_dim, coords, dst_stride, dst_live, op, aux)"},
    {"conv_chw", (PyCFunction)(void (*)(void))conv_chw, METH_FASTCALL,
     "conv_chw(native, group_m, split_k, X, xshape, W, stride, pad, dil, view, shape, bsum)"},
    {"stream", current_stream, METH_NOARGS, "handle of torch's current stream"},
    {nullptr, nullptr, 0, nullptr}};

PyModuleDef module_def = {PyModuleDef_HEAD_INIT, "_hrn_torch", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__hrn_torch(void) { return PyModule_Create(&module_def); }
