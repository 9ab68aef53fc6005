// The host side of one call, from tensors to mmx_gemm_splitk, mmx_gemm_unpacked, mmx_matvec or the packing and quantising
// entry points, as CPython functions (module mm_amx_amd._host_call).
//
// What bounds a small product is the host: the same checks as Python statements, the descriptor as a ctypes structure, the query
// of the workspace and the call through ctypes took 9.7 us for 256 x 256 x 256, under 4 us of which are on the device; 4.7 now.
// (One decode row over 512 x 512 int4 weights 9.2 -> 4.2, a 64 x 512 x 512 layer with a bias 10.2 -> 5.2.)  The functions below
// take the calls that are regular in every respect - tensors of exactly torch's own type on one GPU, the current one, everything
// large enough - and leave all others to the Python form (they return None, and have done nothing), which accepts them or says
// what is wrong.  They keep nothing from one call for the next.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <ATen/ops/empty.h>
#include <torch/csrc/autograd/python_variable.h>

#include "../../include/mm_amx_amd.h"

namespace {

using gemm_fn = decltype(&mmx_gemm_splitk);
using need_fn = decltype(&mmx_gemm_workspace_bytes);
using unpacked_fn = decltype(&mmx_gemm_unpacked);
using unpacked_need_fn = decltype(&mmx_gemm_unpacked_workspace_bytes);
using matvec_fn = decltype(&mmx_matvec);
gemm_fn call_gemm = nullptr;  // of the library that the package has loaded, set once
need_fn call_need = nullptr;
unpacked_fn call_unpacked = nullptr;
unpacked_need_fn call_unpacked_need = nullptr;
matvec_fn call_matvec = nullptr;
decltype(&mmx_packed_b_bytes) call_packed_bytes = nullptr;
decltype(&mmx_repack_b) call_repack = nullptr;
decltype(&mmx_quantize_weights_scratch) call_quantize = nullptr;
decltype(&mmx_quantize_weights_scaled) call_quantize_scaled = nullptr;
decltype(&mmx_quantize_pack_int4) call_quantize_int4 = nullptr;
decltype(&mmx_quantize_pack_scaled) call_quantize_pack_scaled = nullptr;

struct Leave {};  // not a regular call

bool whole_number(PyObject* o, long long lo, long long hi, int& v) {
    if (!PyLong_CheckExact(o)) return false;
    int over = 0;
    const long long x = PyLong_AsLongLongAndOverflow(o, &over);
    if (over || x < lo || x > hi) return false;
    v = (int)x;
    return true;
}

int code_of(at::ScalarType t) {
    switch (t) {
    case at::kFloat: return MMX_F32;
    case at::kBFloat16: return MMX_BF16;
    case at::kChar: return MMX_I8;
    case at::kInt: return MMX_I32;
    case at::kByte: return MMX_U8;
    default: return -1;
    }
}

const at::Tensor& tensor_on(PyObject* o, int device) {
    if (!THPVariable_CheckExact(o)) throw Leave();
    const at::Tensor& t = THPVariable_Unpack(o);
    if (!t.is_cuda() || t.get_device() != device || t.layout() != at::kStrided) throw Leave();
    return t;
}

// a matrix whose elements of a row follow each other; of a single row or column torch leaves the other stride arbitrary
int64_t row_stride_bytes(const at::Tensor& t) {
    if (t.dim() != 2 || (t.stride(1) != 1 && t.size(1) != 1)) throw Leave();
    return (t.size(0) == 1 ? t.size(1) : t.stride(0)) * (int64_t)t.element_size();
}

const float* column_operand(PyObject* o, int device, int n1) {
    if (o == Py_None) return nullptr;
    const at::Tensor& t = tensor_on(o, device);
    if (t.scalar_type() != at::kFloat || !t.is_contiguous() || t.numel() < n1) throw Leave();
    return static_cast<const float*>(t.mutable_data_ptr());
}

void* stream_of(PyObject* o) {
    void* const stream = PyLong_AsVoidPtr(o);
    if (!stream && PyErr_Occurred()) {
        PyErr_Clear();
        throw Leave();
    }
    return stream;
}

// a: C, steps, bias, deq, deq_per_oc, q, q_per_oc; C holds the M x n1 result (half the columns with SILU_GATE)
mmx_epilogue epilogue_of(PyObject* const* a, int device, int64_t M, int n1) {
    const at::Tensor& C = tensor_on(a[0], device);
    int steps;
    if (!whole_number(a[1], 0, INT32_MAX, steps) || !PyFloat_CheckExact(a[3]) || !PyFloat_CheckExact(a[5])) throw Leave();
    mmx_epilogue e = {};
    e.steps = (uint32_t)steps;
    e.out_dtype = code_of(C.scalar_type());
    e.ldc_bytes = row_stride_bytes(C);
    if (e.out_dtype < 0 || C.size(0) < M || C.size(1) < ((steps & MMX_PP_SILU_GATE) ? n1 / 2 : n1)) throw Leave();
    e.C = C.mutable_data_ptr();
    e.bias = column_operand(a[2], device, n1);
    e.deq_scale = (float)PyFloat_AS_DOUBLE(a[3]);
    e.deq_scale_per_oc = column_operand(a[4], device, n1);
    e.q_scale = (float)PyFloat_AS_DOUBLE(a[5]);
    e.q_scale_per_oc = column_operand(a[6], device, n1);
    return e;
}

// gemm(A, Bpacked, N, b_dtype, n0, n1, k_splits, ws, device, stream, C, steps, bias, deq, deq_per_oc, q, q_per_oc)
//   b_dtype: None = that of A; n1: None = N; ws: None = unsplit if the call has no use for one
PyObject* gemm(PyObject*, PyObject* const* a, Py_ssize_t count) {
    if (count != 17 || !call_gemm) Py_RETURN_NONE;
    int rc;
    try {
        int N, n0, n1, ks, device, b_dt;
        if (!whole_number(a[8], 0, 1 << 20, device) || !whole_number(a[2], 1, INT32_MAX, N)) throw Leave();
        n1 = N;
        if (a[5] != Py_None && !whole_number(a[5], 1, N, n1)) throw Leave();
        if (!whole_number(a[4], 0, n1 - 1, n0) || !whole_number(a[6], 0, 1 << 20, ks)) throw Leave();
        const at::Tensor &A = tensor_on(a[0], device), &B = tensor_on(a[1], device);
        const int64_t lda = row_stride_bytes(A), M = A.size(0), K = A.size(1);
        const int a_dt = code_of(A.scalar_type());
        if (M < 1 || M > INT32_MAX || K < 1 || K > INT32_MAX || (a_dt != MMX_BF16 && a_dt != MMX_I8)) throw Leave();
        b_dt = a_dt;
        if (a[3] != Py_None && !whole_number(a[3], 0, 255, b_dt)) throw Leave();
        if (b_dt != MMX_BF16 && b_dt != MMX_I8 && b_dt != MMX_I4) throw Leave();
        // everything that the kernels take on trust: what is too small is an error, and the Python form says which
        const int64_t panels = ((int64_t)N + 31) / 32;
        const int64_t need = b_dt == MMX_I4 ? panels * ((K + 255) / 256 * 4) * 1024 : panels * 32 * ((K * (b_dt == MMX_BF16 ? 2 : 1) + 127) / 128 * 128);
        if (B.scalar_type() != at::kByte || !B.is_contiguous() || B.numel() < need) throw Leave();
        const mmx_epilogue e = epilogue_of(a + 10, device, M, n1);
        void* ws = nullptr;
        size_t ws_bytes = 0;
        if (a[7] != Py_None) {
            const at::Tensor& w = tensor_on(a[7], device);
            if (w.scalar_type() != at::kByte || !w.is_contiguous()) throw Leave();
            ws = w.mutable_data_ptr();
            ws_bytes = (size_t)w.numel();
        } else if (ks != 1) {
            // an explicit count of slices, or a first call that has a use for a workspace: it is made outside
            if (ks || call_need(a_dt, b_dt, (int)M, (int)K, N, n0, n1, e.steps, 0)) throw Leave();
            ks = 1;
        }
        void* const stream = stream_of(a[9]);
        const void *pa = A.mutable_data_ptr(), *pb = B.mutable_data_ptr();
        Py_BEGIN_ALLOW_THREADS
        rc = call_gemm(a_dt, b_dt, pa, lda, pb, (int)M, (int)K, N, n0, n1, &e, ks, ws, ws_bytes, stream);
        Py_END_ALLOW_THREADS
    } catch (...) {  // (tensors without memory of their own throw when asked for it)
        Py_RETURN_NONE;
    }
    return PyLong_FromLong(rc);
}

// gemm_unpacked(A, B, transpose, ws, device, stream, C, steps, bias, deq, deq_per_oc, q, q_per_oc): a B that is used once, where
// the library reads it in place
PyObject* gemm_unpacked(PyObject*, PyObject* const* a, Py_ssize_t count) {
    if (count != 13 || !call_unpacked) Py_RETURN_NONE;
    int rc;
    try {
        int device;
        if (!whole_number(a[4], 0, 1 << 20, device) || !PyBool_Check(a[2])) throw Leave();
        const int transpose = a[2] == Py_True;
        const at::Tensor &A = tensor_on(a[0], device), &B = tensor_on(a[1], device);
        const int64_t lda = row_stride_bytes(A), ldb = row_stride_bytes(B), M = A.size(0), K = A.size(1), N = B.size(transpose ? 0 : 1);
        if (A.scalar_type() != at::kBFloat16 || B.scalar_type() != at::kBFloat16 || B.size(transpose ? 1 : 0) != K) throw Leave();
        if (M < 1 || M > INT32_MAX || K < 1 || K > INT32_MAX || N < 1 || N > INT32_MAX) throw Leave();
        const int64_t need = call_unpacked_need(MMX_BF16, (int)M, (int)K, (int)N, lda, ldb, transpose);
        if (need < 0) throw Leave();
        const mmx_epilogue e = epilogue_of(a + 6, device, M, (int)N);
        if (e.steps & MMX_PP_SILU_GATE) throw Leave();
        const char *pa = static_cast<const char*>(A.mutable_data_ptr()), *pb = static_cast<const char*>(B.mutable_data_ptr()), *pc = static_cast<const char*>(e.C);
        // (a result that is written over B is not computed from B in place)
        if (pc < pb + (B.size(0) - 1) * ldb + 2 * B.size(1) && pb < pc + (M - 1) * e.ldc_bytes + N * (e.out_dtype == MMX_BF16 ? 2 : (e.out_dtype == MMX_I8 ? 1 : 4))) throw Leave();
        void* ws = nullptr;
        size_t ws_bytes = 0;
        if (need) {
            const at::Tensor& w = tensor_on(a[3], device);
            if (w.numel() < need) throw Leave();  // (it is made outside)
            ws = w.mutable_data_ptr();
            ws_bytes = (size_t)w.numel();
        }
        void* const stream = stream_of(a[5]);
        Py_BEGIN_ALLOW_THREADS
        rc = call_unpacked(MMX_BF16, pa, lda, pb, ldb, transpose, (int)M, (int)K, (int)N, &e, ws, ws_bytes, stream);
        Py_END_ALLOW_THREADS
    } catch (...) {
        Py_RETURN_NONE;
    }
    return PyLong_FromLong(rc);
}

// matvec(A, b, out, device, stream)
PyObject* matvec(PyObject*, PyObject* const* a, Py_ssize_t count) {
    if (count != 5 || !call_matvec) Py_RETURN_NONE;
    int rc;
    try {
        int device;
        if (!whole_number(a[3], 0, 1 << 20, device)) throw Leave();
        const at::Tensor &A = tensor_on(a[0], device), &b = tensor_on(a[1], device), &c = tensor_on(a[2], device);
        const int64_t lda = row_stride_bytes(A), M = A.size(0), K = A.size(1);
        const int dt = code_of(A.scalar_type());
        if (M < 1 || M > INT32_MAX || K < 1 || K > INT32_MAX || (dt != MMX_BF16 && dt != MMX_I8)) throw Leave();
        if (b.scalar_type() != A.scalar_type() || b.numel() != K || !b.is_contiguous()) throw Leave();
        if (c.scalar_type() != (dt == MMX_BF16 ? at::kFloat : at::kInt) || c.numel() < M || !c.is_contiguous()) throw Leave();
        const void *pa = A.mutable_data_ptr(), *pb = b.mutable_data_ptr();
        void *pc = c.mutable_data_ptr(), *stream = stream_of(a[4]);
        Py_BEGIN_ALLOW_THREADS
        rc = call_matvec(dt, pa, lda, pb, pc, (int)M, (int)K, stream);
        Py_END_ALLOW_THREADS
    } catch (...) {
        Py_RETURN_NONE;
    }
    return PyLong_FromLong(rc);
}

// ---- packing and quantising: results are made here; an error of the library comes back as its number -------------------
// f() with the interpreter's lock released, as torch's own calls and ctypes have it; what it throws (no memory
// left, say) is left to the Python form, which then says so
template <typename F>
bool unlocked(F&& f) {
    bool ok = true;
    PyThreadState* const state = PyEval_SaveThread();
    try {
        f();
    } catch (...) {
        ok = false;
    }
    PyEval_RestoreThread(state);
    return ok;
}

at::Tensor make(at::IntArrayRef sizes, at::ScalarType type, const at::Tensor& like) {
    return at::empty(sizes, at::TensorOptions().dtype(type).device(like.device()));
}

struct Matrix {
    const at::Tensor* t;
    int64_t ld;
    int rows, cols;
    const void* data;
};
Matrix matrix(PyObject* o, int device) {
    const at::Tensor& t = tensor_on(o, device);
    const int64_t ld = row_stride_bytes(t);
    if (t.size(0) < 1 || t.size(0) > INT32_MAX || t.size(1) < 1 || t.size(1) > INT32_MAX) throw Leave();
    return {&t, ld, (int)t.size(0), (int)t.size(1), t.mutable_data_ptr()};
}

// gemm_packing(A, B, transpose, ws, device, stream, C, steps, bias, deq, deq_per_oc, q, q_per_oc) -> packed: a B that is used once, where the
// library would have it packed first
PyObject* gemm_packing(PyObject*, PyObject* const* a, Py_ssize_t count) {
    if (count != 13 || !call_unpacked_need || !call_repack || !call_gemm) Py_RETURN_NONE;
    try {
        int device, rc = 0;
        if (!whole_number(a[4], 0, 1 << 20, device) || !PyBool_Check(a[2])) throw Leave();
        const int transpose = a[2] == Py_True;
        const Matrix A = matrix(a[0], device), B = matrix(a[1], device);
        const int M = A.rows, K = A.cols, N = transpose ? B.rows : B.cols;
        if (A.t->scalar_type() != at::kBFloat16 || B.t->scalar_type() != at::kBFloat16 || (transpose ? B.cols : B.rows) != K) throw Leave();
        if (call_unpacked_need(MMX_BF16, M, K, N, A.ld, B.ld, transpose) >= 0) throw Leave();
        const mmx_epilogue e = epilogue_of(a + 6, device, M, N);
        if (e.steps & MMX_PP_SILU_GATE) throw Leave();
        void* ws = nullptr;
        size_t ws_bytes = 0;
        if (a[3] != Py_None) {
            const at::Tensor& w = tensor_on(a[3], device);
            if (w.scalar_type() != at::kByte || !w.is_contiguous()) throw Leave();
            ws = w.mutable_data_ptr();
            ws_bytes = (size_t)w.numel();
        } else if (call_need(MMX_BF16, MMX_BF16, M, K, N, 0, N, e.steps, 0)) {
            throw Leave();  // (it is made outside)
        }
        void* const stream = stream_of(a[5]);
        at::Tensor out;
        if (!unlocked([&] {
                out = make({(int64_t)call_packed_bytes(MMX_BF16, K, N)}, at::kByte, *B.t);
                rc = call_repack(MMX_BF16, B.data, B.ld, K, N, transpose, out.mutable_data_ptr(), stream);
                if (!rc) rc = call_gemm(MMX_BF16, MMX_BF16, A.data, A.ld, out.mutable_data_ptr(), M, K, N, 0, N, &e, ws ? 0 : 1, ws, ws_bytes, stream);
            })) throw Leave();
        return rc ? PyLong_FromLong(rc) : THPVariable_Wrap(out);
    } catch (...) {
        Py_RETURN_NONE;
    }
}

// repack(B, transpose, device, stream) -> packed
PyObject* repack(PyObject*, PyObject* const* a, Py_ssize_t count) {
    if (count != 4 || !call_repack) Py_RETURN_NONE;
    try {
        int device, rc = 0;
        if (!whole_number(a[2], 0, 1 << 20, device) || !PyBool_Check(a[1])) throw Leave();
        const Matrix B = matrix(a[0], device);
        const int dt = code_of(B.t->scalar_type()), transpose = a[1] == Py_True, K = transpose ? B.cols : B.rows, N = transpose ? B.rows : B.cols;
        if (dt != MMX_BF16 && dt != MMX_I8 && dt != MMX_U8) throw Leave();
        void* const stream = stream_of(a[3]);
        at::Tensor out;
        if (!unlocked([&] {
                out = make({(int64_t)call_packed_bytes(dt, K, N)}, at::kByte, *B.t);
                rc = call_repack(dt, B.data, B.ld, K, N, transpose, out.mutable_data_ptr(), stream);
            })) throw Leave();
        return rc ? PyLong_FromLong(rc) : THPVariable_Wrap(out);
    } catch (...) {
        Py_RETURN_NONE;
    }
}

// quantize(W, device, stream) -> (Wq, scales)
PyObject* quantize(PyObject*, PyObject* const* a, Py_ssize_t count) {
    if (count != 3 || !call_quantize) Py_RETURN_NONE;
    try {
        int device, rc = 0;
        if (!whole_number(a[1], 0, 1 << 20, device)) throw Leave();
        const Matrix W = matrix(a[0], device);
        if (W.t->scalar_type() != at::kBFloat16) throw Leave();
        void* const stream = stream_of(a[2]);
        at::Tensor Wq, scales, scratch;
        if (!unlocked([&] {
                Wq = make({W.rows, W.cols}, at::kChar, *W.t);
                scales = make({2}, at::kFloat, *W.t);
                scratch = make({MMX_QUANTIZE_SCRATCH_BYTES / 4}, at::kInt, *W.t);
                rc = call_quantize(W.data, W.ld, W.rows, W.cols, Wq.mutable_data_ptr(), W.cols, static_cast<float*>(scales.mutable_data_ptr()),
                                   static_cast<uint32_t*>(scratch.mutable_data_ptr()), MMX_QUANTIZE_SCRATCH_BYTES, stream);
            })) throw Leave();
        return rc ? PyLong_FromLong(rc) : Py_BuildValue("(NN)", THPVariable_Wrap(Wq), THPVariable_Wrap(scales));
    } catch (...) {
        Py_RETURN_NONE;
    }
}

// quantize_scaled(W, scale, device, stream) -> Wq
PyObject* quantize_scaled(PyObject*, PyObject* const* a, Py_ssize_t count) {
    if (count != 4 || !call_quantize_scaled) Py_RETURN_NONE;
    try {
        int device, rc = 0;
        if (!whole_number(a[2], 0, 1 << 20, device) || !PyFloat_CheckExact(a[1])) throw Leave();
        const Matrix W = matrix(a[0], device);
        if (W.t->scalar_type() != at::kBFloat16) throw Leave();
        const float scale = (float)PyFloat_AS_DOUBLE(a[1]);
        void* const stream = stream_of(a[3]);
        at::Tensor Wq;
        if (!unlocked([&] {
                Wq = make({W.rows, W.cols}, at::kChar, *W.t);
                rc = call_quantize_scaled(W.data, W.ld, W.rows, W.cols, scale, Wq.mutable_data_ptr(), W.cols, stream);
            })) throw Leave();
        return rc ? PyLong_FromLong(rc) : THPVariable_Wrap(Wq);
    } catch (...) {
        Py_RETURN_NONE;
    }
}

// quantize_pack_scaled(W, scale, device, stream) -> packed
PyObject* quantize_pack_scaled(PyObject*, PyObject* const* a, Py_ssize_t count) {
    if (count != 4 || !call_quantize_pack_scaled) Py_RETURN_NONE;
    try {
        int device, rc = 0;
        if (!whole_number(a[2], 0, 1 << 20, device) || !PyFloat_CheckExact(a[1])) throw Leave();
        const Matrix W = matrix(a[0], device);
        if (W.t->scalar_type() != at::kBFloat16) throw Leave();
        const float scale = (float)PyFloat_AS_DOUBLE(a[1]);
        void* const stream = stream_of(a[3]);
        at::Tensor out;
        if (!unlocked([&] {
                out = make({(int64_t)call_packed_bytes(MMX_I8, W.rows, W.cols)}, at::kByte, *W.t);
                rc = call_quantize_pack_scaled(W.data, W.ld, W.rows, W.cols, scale, out.mutable_data_ptr(), stream);
            })) throw Leave();
        return rc ? PyLong_FromLong(rc) : THPVariable_Wrap(out);
    } catch (...) {
        Py_RETURN_NONE;
    }
}

// quantize_pack_int4(W, transpose, device, stream) -> (packed, deq)
PyObject* quantize_pack_int4(PyObject*, PyObject* const* a, Py_ssize_t count) {
    if (count != 4 || !call_quantize_int4) Py_RETURN_NONE;
    try {
        int device, rc = 0;
        if (!whole_number(a[2], 0, 1 << 20, device) || !PyBool_Check(a[1])) throw Leave();
        const Matrix W = matrix(a[0], device);
        if (W.t->scalar_type() != at::kBFloat16) throw Leave();
        const int transpose = a[1] == Py_True, K = transpose ? W.cols : W.rows, N = transpose ? W.rows : W.cols;
        void* const stream = stream_of(a[3]);
        at::Tensor packed, deq;
        if (!unlocked([&] {
                packed = make({(int64_t)call_packed_bytes(MMX_I4, K, N)}, at::kByte, *W.t);
                deq = make({N}, at::kFloat, *W.t);
                rc = call_quantize_int4(W.data, W.ld, K, N, transpose, packed.mutable_data_ptr(), static_cast<float*>(deq.mutable_data_ptr()), stream);
            })) throw Leave();
        return rc ? PyLong_FromLong(rc) : Py_BuildValue("(NN)", THPVariable_Wrap(packed), THPVariable_Wrap(deq));
    } catch (...) {
        Py_RETURN_NONE;
    }
}

// bind(addresses of the eleven entry points, in the order below)
PyObject* bind(PyObject*, PyObject* const* a, Py_ssize_t count) {
    constexpr int ENTRIES = 11;
    if (count != ENTRIES) {
        PyErr_SetString(PyExc_TypeError, "bind takes eleven addresses");
        return nullptr;
    }
    void* at[ENTRIES];
    for (int i = 0; i < ENTRIES; i++) at[i] = PyLong_AsVoidPtr(a[i]);
    if (PyErr_Occurred()) return nullptr;
    int i = 0;
    auto set = [&](auto& f) { f = reinterpret_cast<std::remove_reference_t<decltype(f)>>(at[i++]); };
    set(call_gemm);
    set(call_need);
    set(call_unpacked);
    set(call_unpacked_need);
    set(call_matvec);
    set(call_packed_bytes);
    set(call_repack);
    set(call_quantize);
    set(call_quantize_scaled);
    set(call_quantize_int4);
    set(call_quantize_pack_scaled);
    Py_RETURN_NONE;
}

#define METHOD(name) {#name, (PyCFunction)(void (*)(void))name, METH_FASTCALL, nullptr}
PyMethodDef methods[] = {METHOD(gemm), METHOD(gemm_unpacked), METHOD(gemm_packing), METHOD(matvec), METHOD(repack), METHOD(quantize), METHOD(quantize_scaled),
                         METHOD(quantize_pack_int4), METHOD(quantize_pack_scaled), METHOD(bind), {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_host_call", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

// torch_version: of the torch that this was compiled against, whose classes may be laid out differently in another
PyMODINIT_FUNC PyInit__host_call(void) {
    PyObject* const m = PyModule_Create(&module);
    if (m && PyModule_AddStringConstant(m, "torch_version", MMX_TORCH_VERSION) < 0) {
        Py_DECREF(m);
        return nullptr;
    }
    return m;
}
