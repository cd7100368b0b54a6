// spmm(), sddmm() and fused() of dlspm_hip.py as native functions: the checks of the arguments, the look-up of the
// current stream and the call of the C ABI, without the interpreter in between. What bounds a call on a small matrix is
// the host: 9 us of Python and ctypes around a launch of 2.5 us and a kernel of 4 us before these functions.
//
// Each takes the arguments of its Python counterpart. Everything that is not the usual case -- an operand that fails a
// check, schedule memory, a bare row or cut plan -- is handed to that counterpart (register_fallbacks), which computes it
// or raises the exception that says what is wrong; the checks here only have to be at least as strict.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <ATen/ATen.h>
#include <ATen/hip/EmptyTensor.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/autograd/python_variable.h>

#include "../../include/dlspm_hip.h"

namespace {

PyObject* g_fallback[3];  // the Python implementations of the three ops, by DLSPM_OP_*
PyObject* g_prepared;     // class Prepared
PyObject* g_raise;        // raises DlspmError(status, where)
PyObject *g_memory, *g_size_and_hints;  // its attributes

const char* const kSpmmArgs[] = {"row_offsets", "col_indices", "values", "B", "K", "out", "workspace", "plan", "banded"};
const char* const kSddmmArgs[] = {"row_offsets", "col_indices", "lhs", "rhs", "out", "workspace", "plan", "banded"};
const char* const kFusedArgs[] = {"row_offsets", "col_indices", "Q", "Kmat", "V", "scale", "out", "workspace", "plan", "banded"};
constexpr int kMostArgs = 10;

// positional and keyword arguments into slots (nullptr: not given, or None where that is the default: from `optional` on);
// false: leave it to the Python implementation
bool collect(PyObject* const* args, Py_ssize_t npos, PyObject* kwnames, const char* const* names, int optional, int count,
             PyObject** slot)
{
    if (npos > count) return false;
    for (int i = 0; i < count; ++i) slot[i] = i < npos ? args[i] : nullptr;
    const Py_ssize_t nkw = kwnames ? PyTuple_GET_SIZE(kwnames) : 0;
    for (Py_ssize_t k = 0; k < nkw; ++k) {
        PyObject* name = PyTuple_GET_ITEM(kwnames, k);
        int i = 0;
        while (i < count && PyUnicode_CompareWithASCIIString(name, names[i]) != 0) ++i;
        if (i == count || slot[i]) return false;
        slot[i] = args[npos + k];
    }
    for (int i = optional; i < count; ++i)
        if (slot[i] == Py_None) slot[i] = nullptr;
    return true;
}

// the tensor behind `object` if it is a contiguous device tensor of this type, else nullptr
const at::Tensor* device_tensor(PyObject* object, at::ScalarType type)
{
    if (!object || !THPVariable_Check(object)) return nullptr;
    const at::Tensor& t = THPVariable_Unpack(object);
    return t.is_cuda() && t.scalar_type() == type && t.is_contiguous() ? &t : nullptr;
}
void* address(const at::Tensor& t) { return t.numel() > 0 ? t.data_ptr() : nullptr; }
constexpr int64_t kMostInt = 0x7fffffff;

// One call's operands that the three ops have in common: the CSR structure, the plan and the result
struct Call {
    int M = 0, nnz = 0;
    const int *row_offsets = nullptr, *col_indices = nullptr;
    void* memory = nullptr;
    size_t size_and_hints = 0;
    at::Tensor scratch;  // memory of this call alone
    PyObject* result = nullptr;  // a new reference
    float* out = nullptr;

    bool structure(PyObject* offsets, PyObject* columns)
    {
        const at::Tensor *ro = device_tensor(offsets, at::kInt), *ci = device_tensor(columns, at::kInt);
        if (!ro || !ci || ro->numel() < 1 || ro->numel() > kMostInt || ci->numel() > kMostInt) return false;
        M = (int)(ro->numel() - 1);
        nnz = (int)ci->numel();
        row_offsets = static_cast<const int*>(address(*ro));
        col_indices = static_cast<const int*>(address(*ci));
        return true;
    }
    // `workspace`, `plan` and `banded`: nothing, or what prepare() returned
    bool plan(PyObject* workspace, PyObject* plan, PyObject* banded)
    {
        if (workspace || (banded && banded != Py_False)) return false;
        if (!plan) return true;
        if ((PyObject*)Py_TYPE(plan) != g_prepared) return false;
        PyObject* mem = PyObject_GetAttr(plan, g_memory);
        PyObject* size = mem ? PyObject_GetAttr(plan, g_size_and_hints) : nullptr;
        bool good = size != nullptr && PyLong_Check(size);
        if (good) size_and_hints = (size_t)PyLong_AsUnsignedLongLong(size);
        if (good && mem != Py_None) {
            good = THPVariable_Check(mem);
            if (good) memory = THPVariable_Unpack(mem).data_ptr();
        }
        if (PyErr_Occurred()) {
            PyErr_Clear();
            good = false;
        }
        Py_XDECREF(mem);
        Py_XDECREF(size);
        return good;
    }
    // What prepare() left to be allocated by each call: from PyTorch's allocator, so that calls on several streams do not share it.
    // Without it, where there is no room, the call runs as with the hints alone.
    void own_memory(const at::Tensor& like)
    {
        const size_t bytes = size_and_hints & ~DLSPM_HINT_MASK;
        if (memory || bytes == 0) return;
        try {
            scratch = at::detail::empty_cuda({(int64_t)bytes}, at::kByte, like.device(), std::nullopt);
            memory = scratch.data_ptr();
        } catch (const c10::OutOfMemoryError&) {
            size_and_hints &= DLSPM_HINT_MASK;
        } catch (...) {
            Py_DECREF(result);
            throw;
        }
    }
    // `given`, or a new tensor on `like`'s device
    bool output(PyObject* given, at::IntArrayRef sizes, const at::Tensor& like)
    {
        int64_t count = 1;
        for (int64_t s : sizes) count *= s;
        if (given) {
            const at::Tensor* t = device_tensor(given, at::kFloat);
            if (!t || t->numel() < count) return false;
            out = static_cast<float*>(address(*t));
            Py_INCREF(given);
            result = given;
        } else {
            // (at::empty without the dispatcher: every element is written by the call)
            at::Tensor t = at::detail::empty_cuda(sizes, at::kFloat, like.device(), std::nullopt);
            out = static_cast<float*>(address(t));
            result = THPVariable_Wrap(std::move(t));
        }
        return result != nullptr;
    }
    template <typename Launch> PyObject* run(const char* where, Launch&& launch)
    {
        void* stream;
        try {  // (before the lock is released: no exception may pass through that block)
            stream = static_cast<void*>(c10::hip::getCurrentHIPStream().stream());
        } catch (...) {
            Py_DECREF(result);
            throw;
        }
        int status;
        Py_BEGIN_ALLOW_THREADS
        status = launch(stream);
        Py_END_ALLOW_THREADS
        if (status == DLSPM_OK) return result;
        Py_DECREF(result);
        return PyObject_CallFunction(g_raise, "is", status, where);
    }
};

PyObject* fallback(int op, PyObject* const* args, Py_ssize_t npos, PyObject* kwnames)
{
    return PyObject_Vectorcall(g_fallback[op], args, (size_t)npos, kwnames);
}

// A result that cannot be allocated is another call for the Python implementation: it raises torch.OutOfMemoryError there.
template <typename Body> PyObject* guarded(int op, PyObject* const* args, Py_ssize_t npos, PyObject* kwnames, Body&& body)
{
    try {
        return body();
    } catch (const c10::OutOfMemoryError&) {
        return fallback(op, args, npos, kwnames);
    } catch (const c10::Error& e) {
        PyErr_SetString(PyExc_RuntimeError, e.what_without_backtrace());
    } catch (const std::exception& e) {
        PyErr_SetString(PyExc_RuntimeError, e.what());
    }
    return nullptr;
}

PyObject* call_spmm(PyObject*, PyObject* const* args, Py_ssize_t npos, PyObject* kwnames)
{
    return guarded(DLSPM_OP_SPMM, args, npos, kwnames, [&]() -> PyObject* {
        PyObject* a[kMostArgs];
        Call c;
        const at::Tensor *values, *B;
        if (!collect(args, npos, kwnames, kSpmmArgs, 4, 9, a) || !c.structure(a[0], a[1]) || !c.plan(a[6], a[7], a[8]) || (a[4] && !PyLong_Check(a[4])) ||
            !(values = device_tensor(a[2], at::kFloat)) || !(B = device_tensor(a[3], at::kFloat)) || B->dim() != 2 ||
            values->numel() < c.nnz || B->size(0) > kMostInt || B->size(1) > kMostInt)
            return fallback(DLSPM_OP_SPMM, args, npos, kwnames);
        const long long K_given = a[4] ? PyLong_AsLongLong(a[4]) : B->size(0);
        if (K_given < 0 || K_given > B->size(0) || !c.output(a[5], {c.M, B->size(1)}, *B)) {
            PyErr_Clear();
            return fallback(DLSPM_OP_SPMM, args, npos, kwnames);
        }
        c.own_memory(*B);
        const int K = (int)K_given, N = (int)B->size(1);
        const float *v = static_cast<const float*>(address(*values)), *b = static_cast<const float*>(address(*B));
        return c.run("spmm_csr_f32", [&](void* stream) {
            return spmm_csr_f32(c.M, K, N, c.nnz, c.row_offsets, c.col_indices, v, b, c.out, c.memory, c.size_and_hints, stream);
        });
    });
}

PyObject* call_sddmm(PyObject*, PyObject* const* args, Py_ssize_t npos, PyObject* kwnames)
{
    return guarded(DLSPM_OP_SDDMM, args, npos, kwnames, [&]() -> PyObject* {
        PyObject* a[kMostArgs];
        Call c;
        const at::Tensor *lhs, *rhs;
        if (!collect(args, npos, kwnames, kSddmmArgs, 4, 8, a) || !c.structure(a[0], a[1]) || !c.plan(a[5], a[6], a[7]) ||
            !(lhs = device_tensor(a[2], at::kFloat)) || !(rhs = device_tensor(a[3], at::kFloat)) || lhs->dim() != 2 ||
            rhs->dim() != 2 || lhs->size(1) != rhs->size(1) || lhs->size(0) < c.M || rhs->size(0) > kMostInt ||
            rhs->size(1) > kMostInt || !c.output(a[4], {c.nnz}, *lhs))
            return fallback(DLSPM_OP_SDDMM, args, npos, kwnames);
        c.own_memory(*lhs);
        const int K = (int)rhs->size(0), D = (int)rhs->size(1);
        const float *l = static_cast<const float*>(address(*lhs)), *r = static_cast<const float*>(address(*rhs));
        return c.run("sddmm_csr_f32", [&](void* stream) {
            return sddmm_csr_f32(c.M, K, D, c.nnz, c.row_offsets, c.col_indices, l, r, c.out, c.memory, c.size_and_hints, stream);
        });
    });
}

PyObject* call_fused(PyObject*, PyObject* const* args, Py_ssize_t npos, PyObject* kwnames)
{
    return guarded(DLSPM_OP_FUSED, args, npos, kwnames, [&]() -> PyObject* {
        PyObject* a[kMostArgs];
        Call c;
        const at::Tensor *Q, *Km, *V;
        if (!collect(args, npos, kwnames, kFusedArgs, 6, 10, a) || !c.structure(a[0], a[1]) || !c.plan(a[7], a[8], a[9]) ||
            !(Q = device_tensor(a[2], at::kFloat)) || !(Km = device_tensor(a[3], at::kFloat)) ||
            !(V = device_tensor(a[4], at::kFloat)) || (a[5] && !PyFloat_Check(a[5])) || Q->dim() != 2 || Km->dim() != 2 ||
            V->sizes() != Km->sizes() || Q->size(1) != Km->size(1) || Q->size(0) < c.M || Km->size(0) > kMostInt ||
            Km->size(1) > kMostInt || !c.output(a[6], {c.M, Km->size(1)}, *Q))
            return fallback(DLSPM_OP_FUSED, args, npos, kwnames);
        c.own_memory(*Q);
        const int K = (int)Km->size(0), D = (int)Km->size(1);
        const float scale = a[5] ? (float)PyFloat_AS_DOUBLE(a[5]) : 1.0f;
        const float *q = static_cast<const float*>(address(*Q)), *k = static_cast<const float*>(address(*Km)),
                    *v = static_cast<const float*>(address(*V));
        return c.run("fused_sddmm_spmm_f32", [&](void* stream) {
            return fused_sddmm_spmm_f32(c.M, K, D, c.nnz, c.row_offsets, c.col_indices, q, k, v, scale, c.out, c.memory,
                                        c.size_and_hints, stream);
        });
    });
}

// register_fallbacks(spmm, sddmm, fused, Prepared, raise_error)
PyObject* register_fallbacks(PyObject*, PyObject* args)
{
    PyObject *f0, *f1, *f2, *prepared, *raise;
    if (!PyArg_ParseTuple(args, "OOOOO", &f0, &f1, &f2, &prepared, &raise)) return nullptr;
    for (PyObject* o : {f0, f1, f2, prepared, raise}) Py_INCREF(o);  // held until the process ends
    g_fallback[DLSPM_OP_SPMM] = f0;
    g_fallback[DLSPM_OP_SDDMM] = f1;
    g_fallback[DLSPM_OP_FUSED] = f2;
    g_prepared = prepared;
    g_raise = raise;
    Py_RETURN_NONE;
}

PyMethodDef kMethods[] = {
    {"register_fallbacks", register_fallbacks, METH_VARARGS, nullptr},
    {"spmm", (PyCFunction)(void*)call_spmm, METH_FASTCALL | METH_KEYWORDS,
     "spmm($module, row_offsets, col_indices, values, B, K=None, out=None, workspace=None, plan=None, banded=False)\n--\n\n"
     "C = A_csr @ B on the current stream (spmm_csr_f32). row_offsets/col_indices int32, values/B float32, all on the GPU.\n"
     "plan: what prepare(), row_plan() or cut_plan() returned. workspace: a GPU tensor of workspace_bytes(OP_SPMM, ...)\n"
     "bytes, or ROWS_EVEN / ROWS_SKEWED. banded: every row's columns lie in a narrow window that moves with the row."},
    {"sddmm", (PyCFunction)(void*)call_sddmm, METH_FASTCALL | METH_KEYWORDS,
     "sddmm($module, row_offsets, col_indices, lhs, rhs, out=None, workspace=None, plan=None, banded=False)\n--\n\n"
     "out[j] = <lhs[i], rhs[col[j]]> for each CSR slot j of row i, on the current stream (sddmm_csr_f32); the options are\n"
     "those of spmm()."},
    {"fused", (PyCFunction)(void*)call_fused, METH_FASTCALL | METH_KEYWORDS,
     "fused($module, row_offsets, col_indices, Q, Kmat, V, scale=1.0, out=None, workspace=None, plan=None, banded=False)\n--\n\n"
     "O = (S .* (Q Kmat^T) * scale) V on the current stream (fused_sddmm_spmm_f32); the scores are not stored, except\n"
     "on dense masks with a plan from prepare(), through memory of the call's own; the options are those of spmm()."},
    {nullptr, nullptr, 0, nullptr}};
PyModuleDef kModule = {PyModuleDef_HEAD_INIT, "_dlspm_torch", nullptr, -1, kMethods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__dlspm_torch(void)
{
    g_memory = PyUnicode_InternFromString("memory");
    g_size_and_hints = PyUnicode_InternFromString("size_and_hints");
    return g_memory && g_size_and_hints ? PyModule_Create(&kModule) : nullptr;
}
