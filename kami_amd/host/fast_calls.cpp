// Native call path of the Python wrappers: checks the tensors of an ordinary call, allocates
// its results and calls the C ABI, without a ctypes call's conversions.
//
// Every function takes the call only when it is plain -- exact torch.Tensor objects on the
// GPU, contiguous (or with unit column stride where the wrapper asks no more), of the right
// types and shapes -- and returns None otherwise, also when the library refuses the call
// before it launches anything or torch cannot give an address: the wrapper then runs its own
// checks, which name what is wrong, and its own call.  An error of the HIP runtime is raised
// from here: work may have been enqueued by then, and a second call would do it twice
// (with beta != 0, add twice).  Nothing is remembered between calls.
#include <algorithm>

#include <torch/csrc/autograd/python_variable.h>

#include <ATen/ATen.h>
#include <c10/hip/HIPStream.h>

#include "../../include/kami.h"
#include "../csrc/spgemm_internal.hpp"

namespace {

// Entry points of the library the Python side has loaded (set by `bind`)
struct Lib {
    decltype(&kami_block_gemm) block_gemm;
    decltype(&kami_split_gemm) split_gemm;
    decltype(&kami_batched_execute) batched_execute;
    decltype(&kami_bsr_spgemm_symbolic) symbolic;
    decltype(&kami_bsr_spgemm_fill) fill;
    decltype(&kami_bsr_spgemm_numeric) numeric;
    decltype(&kami_bsr_spmm) spmm;
    decltype(&kami_bsr_spgemm_structure) structure;
} g_lib;
PyObject* g_check = nullptr;  // check(status, what), raises for a status that is no success
bool g_bound = false;

// Other Python threads run while the library is in a call or torch allocates: a launch waits
// where a stream's queue is full.
struct NoGil {
    PyThreadState* const state = PyEval_SaveThread();
    NoGil() = default;
    NoGil(const NoGil&) = delete;
    ~NoGil() { PyEval_RestoreThread(state); }
};

// What a library call's status means for the native call
struct Refused : std::exception {};      // left to the wrapper
struct PythonError : std::exception {};  // raised: a Python error is set

void done(kami_status st, const char* what) {
    if (st == KAMI_OK) return;
    if (st != KAMI_EHIP) throw Refused();
    PyObject* r = PyObject_CallFunction(g_check, "is", (int)st, what);
    Py_XDECREF(r);
    throw PythonError();
}

void* current_stream() { return c10::hip::getCurrentHIPStream().stream(); }

// The tensor of an exact torch.Tensor on a GPU, or null
const at::Tensor* gpu_tensor(PyObject* o) {
    if (!THPVariable_CheckExact(o)) return nullptr;
    const at::Tensor& t = THPVariable_Unpack(o);
    return t.is_cuda() && t.layout() == at::kStrided ? &t : nullptr;
}

bool is(const at::Tensor& t, at::ScalarType type, const at::Tensor& with) {
    return t.scalar_type() == type && t.device() == with.device();
}

// Input and result types of a precision; false for one the wrappers do not know
bool types_of(int prec, at::ScalarType* in, at::ScalarType* out) {
    switch (prec) {
        case KAMI_PREC_F64:
        case KAMI_PREC_F64_SPLIT_F16:
        case KAMI_PREC_F64_SPLIT_BF16:
        case KAMI_PREC_F64_SPLIT_I8: *in = *out = at::kDouble; return true;
        case KAMI_PREC_F16_F32: *in = at::kHalf; *out = at::kFloat; return true;
        case KAMI_PREC_BF16_F32: *in = at::kBFloat16; *out = at::kFloat; return true;
    }
    return false;
}

int precision_of(const at::Tensor& t) {
    switch (t.scalar_type()) {
        case at::kDouble: return KAMI_PREC_F64;
        case at::kHalf: return KAMI_PREC_F16_F32;
        case at::kBFloat16: return KAMI_PREC_BF16_F32;
        default: return -1;
    }
}

// The wrapper's `precision` argument for a call on `t`; false when it is no precision
bool precision_arg(PyObject* o, const at::Tensor& t, int* prec) {
    if (o == Py_None) {
        *prec = precision_of(t);
        return true;
    }
    const long v = PyLong_AsLong(o);
    if ((v == -1 && PyErr_Occurred()) || v < KAMI_PREC_F64 || v > KAMI_PREC_F64_SPLIT_I8) return false;
    *prec = (int)v;
    return true;
}

// Runs `f`; a torch error (no storage, out of memory) leaves the call to the wrapper
template <class F>
PyObject* plain(F f) {
    if (!g_bound) Py_RETURN_NONE;
    try {
        if (PyObject* r = f()) return r;
    } catch (const PythonError&) {
        if (PyErr_Occurred()) return nullptr;
    } catch (const std::exception&) {
    }
    if (PyErr_Occurred()) PyErr_Clear();
    Py_RETURN_NONE;
}

PyObject* wrap(const at::Tensor& t) { return THPVariable_Wrap(t); }

// block_gemm(A, B, C or None, precision or None, partition, ranks, b_layout, iters, alpha, beta,
//            slices, pipeline, tiled)
PyObject* block_gemm(PyObject*, PyObject* const* a, Py_ssize_t n) {
    return plain([&]() -> PyObject* {
        if (n != 13) return nullptr;
        const at::Tensor *A = gpu_tensor(a[0]), *B = gpu_tensor(a[1]);
        if (!A || !B) return nullptr;
        const int64_t dim = A->dim();
        if ((dim != 2 && dim != 3) || B->dim() != dim) return nullptr;
        kami_gemm_desc d = {};
        int prec;
        if (!precision_arg(a[3], *A, &prec)) return nullptr;
        long v[7];
        const int at_[7] = {4, 5, 6, 7, 10, 11, 12};
        for (int i = 0; i < 7; ++i) {
            v[i] = PyLong_AsLong(a[at_[i]]);
            if (v[i] == -1 && PyErr_Occurred()) return nullptr;
            if (v[i] < INT32_MIN || v[i] > INT32_MAX) return nullptr;
        }
        d.alpha = PyFloat_AsDouble(a[8]);
        d.beta = PyFloat_AsDouble(a[9]);
        if (PyErr_Occurred()) return nullptr;
        at::ScalarType in, out;
        if (!types_of(prec, &in, &out)) return nullptr;
        const int64_t count = dim == 3 ? A->size(0) : 1;
        const int64_t m = A->size(dim - 2), k = A->size(dim - 1);
        const bool kn = v[2] == KAMI_B_KN;
        const int64_t nn = B->size(kn ? dim - 1 : dim - 2);
        if (B->size(kn ? dim - 2 : dim - 1) != k || (dim == 3 && B->size(0) != count)) return nullptr;
        if (m > INT32_MAX || nn > INT32_MAX || k > INT32_MAX) return nullptr;
        if (!is(*A, in, *A) || !is(*B, in, *A) || !A->is_contiguous() || !B->is_contiguous()) return nullptr;
        at::Tensor C;
        if (a[2] != Py_None) {
            const at::Tensor* c = gpu_tensor(a[2]);
            if (!c || c->dim() != dim || !is(*c, out, *A) || !c->is_contiguous()) return nullptr;
            if (c->size(dim - 2) != m || c->size(dim - 1) != nn || (dim == 3 && c->size(0) != count))
                return nullptr;
            C = *c;
        }
        d.m = (int32_t)m;
        d.n = (int32_t)nn;
        d.k = (int32_t)k;
        d.precision = prec;
        d.partition = (int32_t)v[0];
        d.ranks = (int32_t)v[1];
        d.b_layout = (int32_t)v[2];
        d.iters = (int32_t)v[3];
        d.slices = (int32_t)v[4];
        d.pipeline = (int32_t)v[5];
        kami_status st;
        {
            const NoGil released;
            if (!C.defined())
                C = dim == 3 ? at::empty({count, m, nn}, A->options().dtype(out))
                             : at::empty({m, nn}, A->options().dtype(out));
            st = (v[6] ? g_lib.split_gemm : g_lib.block_gemm)(
                &d, A->data_ptr(), B->data_ptr(), C.data_ptr(), count, 0, 0, 0, current_stream());
        }
        done(st, v[6] ? "kami_split_gemm" : "kami_block_gemm");
        if (a[2] == Py_None) return wrap(C);
        Py_INCREF(a[2]);
        return a[2];
    });
}

// batched_execute(plan handle)
PyObject* batched_execute(PyObject*, PyObject* arg) {
    return plain([&]() -> PyObject* {
        void* plan = PyLong_AsVoidPtr(arg);
        if (!plan) return nullptr;
        kami_status st;
        {
            const NoGil released;
            st = g_lib.batched_execute(static_cast<kami_batched_plan*>(plan), current_stream());
        }
        done(st, "kami_batched_execute");
        Py_RETURN_TRUE;
    });
}

// A BSR matrix from (mb, nb, bs, rowptr, colidx, vals); false when it is not plain
bool bsr_of(PyObject* const* a, kami_bsr* X, const at::Tensor* (&t)[3]) {
    const long mb = PyLong_AsLong(a[0]), nb = PyLong_AsLong(a[1]), bs = PyLong_AsLong(a[2]);
    if (PyErr_Occurred()) return false;
    if (mb < 0 || nb < 0 || bs < 0 || mb >= INT32_MAX || nb > INT32_MAX || bs > INT32_MAX) return false;
    for (int i = 0; i < 3; ++i)
        if (!(t[i] = gpu_tensor(a[3 + i])) || !t[i]->is_contiguous() || t[i]->device() != t[0]->device())
            return false;
    const int64_t nnzb = t[1]->numel();
    if (t[0]->scalar_type() != at::kInt || t[0]->dim() != 1 || t[0]->size(0) != mb + 1) return false;
    if (t[1]->scalar_type() != at::kInt || t[1]->dim() != 1 || nnzb > INT32_MAX || nnzb == 0) return false;
    if (t[2]->dim() != 3 || t[2]->size(0) != nnzb || t[2]->size(1) != bs || t[2]->size(2) != bs) return false;
    *X = kami_bsr{(int32_t)mb, (int32_t)nb, (int32_t)bs, (int32_t)nnzb,
                  static_cast<const int32_t*>(t[0]->data_ptr()), static_cast<const int32_t*>(t[1]->data_ptr()),
                  t[2]->data_ptr()};
    return true;
}

// bsr_spmm(6 of A, B, C or None, b_layout, precision or None, alpha, beta)
PyObject* bsr_spmm(PyObject*, PyObject* const* a, Py_ssize_t n) {
    return plain([&]() -> PyObject* {
        kami_bsr A;
        const at::Tensor* t[3];
        if (n != 12 || !bsr_of(a, &A, t)) return nullptr;
        const at::Tensor* B = gpu_tensor(a[6]);
        const long lay = PyLong_AsLong(a[8]);
        const double alpha = PyFloat_AsDouble(a[10]), beta = PyFloat_AsDouble(a[11]);
        int prec;
        if (PyErr_Occurred() || !precision_arg(a[9], *t[2], &prec)) return nullptr;
        at::ScalarType in, out;
        if ((prec != KAMI_PREC_F64 && prec != KAMI_PREC_F16_F32 && prec != KAMI_PREC_BF16_F32) ||
            !types_of(prec, &in, &out))
            return nullptr;
        const bool kn = lay == KAMI_B_KN;
        if (!B || B->dim() != 2 || B->stride(1) != 1 || !is(*B, in, *t[0]) || t[2]->scalar_type() != in) return nullptr;
        const int64_t nn = B->size(kn ? 1 : 0), rows = (int64_t)A.mb * A.bs;
        if (B->size(kn ? 0 : 1) != (int64_t)A.nb * A.bs || nn > INT32_MAX) return nullptr;
        at::Tensor C;
        if (a[7] != Py_None) {
            const at::Tensor* c = gpu_tensor(a[7]);
            if (!c || c->dim() != 2 || !is(*c, out, *B) || c->size(0) != rows || c->size(1) != nn || c->stride(1) != 1)
                return nullptr;
            C = *c;
        }
        kami_status st;
        {
            const NoGil released;
            if (!C.defined()) C = at::zeros({rows, nn}, B->options().dtype(out));
            st = g_lib.spmm(&A, B->data_ptr(), (int32_t)nn, B->stride(0), (int32_t)lay, C.data_ptr(), C.stride(0),
                            prec, alpha, beta, current_stream());
        }
        done(st, "kami_bsr_spmm");
        if (a[7] == Py_None) return wrap(C);
        Py_INCREF(a[7]);
        return a[7];
    });
}

// Columns that may be allocated before nnzb(C) is known whatever C will have: 64 KiB.
constexpr int64_t kRoom = 1 << 14;

// bsr_spgemm(6 of A, 6 of B, precision or None, alpha) -> (rowptr, colidx, vals)
PyObject* bsr_spgemm(PyObject*, PyObject* const* a, Py_ssize_t n) {
    return plain([&]() -> PyObject* {
        kami_bsr A, B;
        const at::Tensor *ta[3], *tb[3];
        if (n != 14 || !bsr_of(a, &A, ta) || !bsr_of(a + 6, &B, tb)) return nullptr;
        const double alpha = PyFloat_AsDouble(a[13]);
        int prec;
        if (PyErr_Occurred() || !precision_arg(a[12], *ta[2], &prec)) return nullptr;
        at::ScalarType in, out;
        if ((prec != KAMI_PREC_F64 && prec != KAMI_PREC_F16_F32 && prec != KAMI_PREC_BF16_F32) ||
            !types_of(prec, &in, &out))
            return nullptr;
        if (A.nb != B.mb || A.bs != B.bs || !is(*ta[2], in, *ta[0]) || !is(*tb[2], in, *ta[0])) return nullptr;
        size_t ws_bytes = (size_t)A.mb * (((size_t)B.nb + 31) / 32) * 4;
        // Up to 2^18 blocks that C could have: the columns are written before the count is known
        // here, and the scan is not a launch of its own.  There is room for all of them up to
        // kRoom, else for twice the products that equal rows would give (8192^2, 2 % of 32 x 32
        // blocks: 13000 of 65536; C has 6606).
        const int64_t most = (int64_t)A.mb * B.nb;
        const bool fused = A.mb <= kStructureRows && most <= (1 << 18);
        const int64_t room = std::min(most, std::max<int64_t>(kRoom, 2 * (int64_t)A.nnzb * B.nnzb / B.mb));
        if (fused) ws_bytes += (size_t)A.mb * 4;
        const auto ints = ta[0]->options();
        at::Tensor rowptr, colidx, vals;
        int64_t nnz = 0;
        kami_status st;
        const char* phase = "kami_bsr_spgemm_symbolic";
        {
            const NoGil released;
            at::Tensor ws = at::empty({(int64_t)ws_bytes / 4}, ints);
            rowptr = at::empty({(int64_t)A.mb + 1}, ints);
            int32_t* const rp = static_cast<int32_t*>(rowptr.data_ptr());
            void* const stream = current_stream();
            if (fused) colidx = at::empty({room}, ints);
            st = fused ? g_lib.structure(&A, &B, rp, static_cast<int32_t*>(colidx.data_ptr()), room, &nnz,
                                         ws.data_ptr(), ws_bytes, stream)
                       : g_lib.symbolic(&A, &B, rp, &nnz, ws.data_ptr(), ws_bytes, stream);
            // kept where C, for as long as it lives, holds no more than kRoom columns or an eighth
            // of its own size too much; written again otherwise, as where the room did not do
            const int64_t block_bytes = (int64_t)A.bs * A.bs * at::elementSize(out) + 4;
            const bool keep = fused && nnz <= room && room - nnz <= std::max(kRoom, nnz * block_bytes / 32);
            if (st == KAMI_OK && keep) {  // the storage's size too, so that a saved C holds its own blocks only
                colidx.unsafeGetTensorImpl()->set_sizes_contiguous({nnz > 0 ? nnz : 1});
                colidx.storage().unsafeGetStorageImpl()->set_nbytes((size_t)(nnz > 0 ? nnz : 1) * 4);
            } else if (st == KAMI_OK) {
                colidx = at::empty({nnz > 0 ? nnz : 1}, ints);
                phase = "kami_bsr_spgemm_fill";
                st = g_lib.fill(&A, &B, rp, static_cast<int32_t*>(colidx.data_ptr()), ws.data_ptr(), ws_bytes, stream);
            }
            if (st == KAMI_OK) {
                vals = at::empty({nnz > 0 ? nnz : 1, A.bs, A.bs}, ta[2]->options().dtype(out));
                phase = "kami_bsr_spgemm_numeric";
                if (nnz > 0)
                    st = g_lib.numeric(&A, &B, rp, static_cast<const int32_t*>(colidx.data_ptr()), nnz,
                                       vals.data_ptr(), prec, alpha, stream);
            }
        }
        done(st, phase);
        if (nnz == 0) {
            colidx = colidx.slice(0, 0, 0);
            vals = vals.slice(0, 0, 0);
        }
        PyObject *r = wrap(rowptr), *c = wrap(colidx), *w = wrap(vals);
        PyObject* res = r && c && w ? PyTuple_Pack(3, r, c, w) : nullptr;
        Py_XDECREF(r);
        Py_XDECREF(c);
        Py_XDECREF(w);
        return res;
    });
}

// bind(check, addresses of the eight entry points, in Lib's order)
PyObject* bind(PyObject*, PyObject* const* a, Py_ssize_t n) {
    void* p[8];
    if (n != 9 || !PyCallable_Check(a[0])) {
        PyErr_SetString(PyExc_TypeError, "bind expects a callable and eight addresses");
        return nullptr;
    }
    for (int i = 0; i < 8; ++i) {
        p[i] = PyLong_AsVoidPtr(a[1 + i]);
        if (!p[i]) {
            if (!PyErr_Occurred()) PyErr_SetString(PyExc_ValueError, "null entry point");
            return nullptr;
        }
    }
    g_lib = Lib{(decltype(Lib::block_gemm))p[0], (decltype(Lib::split_gemm))p[1],
                (decltype(Lib::batched_execute))p[2], (decltype(Lib::symbolic))p[3],
                (decltype(Lib::fill))p[4], (decltype(Lib::numeric))p[5], (decltype(Lib::spmm))p[6],
                (decltype(Lib::structure))p[7]};
    Py_INCREF(a[0]);
    Py_XSETREF(g_check, a[0]);
    g_bound = true;
    Py_RETURN_NONE;
}

PyMethodDef methods[] = {
    {"bind", (PyCFunction)(void*)bind, METH_FASTCALL, nullptr},
    {"block_gemm", (PyCFunction)(void*)block_gemm, METH_FASTCALL, nullptr},
    {"batched_execute", batched_execute, METH_O, nullptr},
    {"bsr_spmm", (PyCFunction)(void*)bsr_spmm, METH_FASTCALL, nullptr},
    {"bsr_spgemm", (PyCFunction)(void*)bsr_spgemm, METH_FASTCALL, nullptr},
    {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_fast_calls", nullptr, -1, methods};

}  // namespace

PyMODINIT_FUNC PyInit__fast_calls() { return PyModule_Create(&module); }
