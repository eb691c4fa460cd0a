// The plain calls of chadslab_amd.ops (qlinear, moe_ffn) from the Python object to the C ABI in one native function.
//
// What bounds a small call is the host: a product of 2048 x 2048 on one token takes 2.9 us on the GPU and took 7.2 us of Python
// (attribute look-ups, checks, the result's allocation, eight arguments through ctypes), a mixture of experts with sixteen experts
// 59 us (96 tensors looked at one by one).  Here the same checks are C++: 4.9 us, and 28 us with the GPU the slower side.
//
// Only what needs nothing unusual is served: exact torch.Tensor objects on the current device, of the right types and shapes,
// contiguous.  For everything else, also for a call whose arguments the library refuses, the functions return None before anything has
// been launched, and the Python code behind them does what it always did: copies, casts, and the errors' texts.  An error of the
// device or of a launch is raised here and now, with the library's text: kernels of the call may be queued, and a second attempt
// would find another error than the one that was reported.
#include <ATen/ops/empty.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/Dtype.h>
#include <torch/csrc/autograd/python_variable.h>

#include "../../include/chadq.h"

namespace {

typedef int (*product_fn)(const void *, const void *, const void *, void *, int, int, int, void *);
typedef size_t (*product_bytes_fn)(int, int, int, int);
typedef int (*product_ws_fn)(const void *, const void *, const void *, void *, int, int, int, void *, size_t, void *);
typedef int (*decode_ws_fn)(const void *, const void *, const void *, void *, int, int, int, int, void *, size_t, void *);
typedef size_t (*moe_bytes_fn)(int, int, int, int, int);
typedef int (*moe_fn)(const void *, const void *, const chadq_moe_expert_i4g32 *, void *, int, int, int, int, int, int, void *, size_t, void *);

enum Entry { GEMV_I4, GEMV_I4_BF16, GEMM_I4, GEMV_I8, GEMV_I8_BF16, GEMM_I8, GEMM_BYTES, GEMM_I4_WS, GEMM_I8_WS, GEMV_BYTES, GEMV_I4_WS, GEMV_I8_WS, MOE_BYTES, MOE_ROWS, MOE_TILES, ENTRIES };
const char *const kEntryNames[ENTRIES] = {"chadq_gemv_i4g32", "chadq_gemv_i4g32_bf16", "chadq_gemm_i4g32_bf16", "chadq_gemv_i8row", "chadq_gemv_i8row_bf16",
                                          "chadq_gemm_i8row_bf16", "chadq_gemm_bf16_workspace_bytes", "chadq_gemm_i4g32_bf16", "chadq_gemm_i8row_bf16",
                                          "chadq_gemv_workspace_bytes", "chadq_gemv_i4g32", "chadq_gemv_i8row", "chadq_moe_ffn_i4g32_workspace_bytes", "chadq_moe_ffn_i4g32",
                                          "chadq_moe_ffn_i4g32_tiled"};
void *g_entry[ENTRIES];                                // of the library in use (bind)
PyObject *g_int4 = nullptr, *g_int8 = nullptr, *g_tiles = nullptr;  // the weight containers
PyObject *g_check = nullptr;                           // _lib.check(status, name): raises
PyObject *s_packed, *s_scale, *s_w;
constexpr int kGemvRows = 16, kMaxExperts = 16;

// a dense GPU tensor that may be handed on as it is
const at::Tensor *plain(PyObject *o, at::ScalarType type, int dim, int device) {
    if (!o || !THPVariable_CheckExact(o)) return nullptr;
    const at::Tensor &t = THPVariable_Unpack(o);
    const c10::TensorImpl *const i = t.unsafeGetTensorImpl();
    if (t.layout() != at::kStrided || !i->has_storage() || !t.is_cuda() || t.dim() != dim || t.scalar_type() != type || !t.is_contiguous() ||
        t.get_device() != device || t.is_neg() || i->is_python_dispatch())
        return nullptr;
    return &t;
}

struct Ref {  // a new reference, dropped at the end of the scope
    PyObject *p;
    explicit Ref(PyObject *o) : p(o) {
        if (!o) PyErr_Clear();
    }
    ~Ref() { Py_XDECREF(p); }
    Ref(const Ref &) = delete;
};

// The interpreter lock is given up for as long as this lives, as torch.empty and ctypes do: an allocation may wait for the device (the
// allocator gives cached memory back and asks again) or run a hook that wants the lock on a thread that another allocation waits for.
struct WithoutLock {
    PyThreadState *const state = PyEval_SaveThread();
    ~WithoutLock() { PyEval_RestoreThread(state); }
};

// What becomes of a call that did not succeed (the text of the error belongs to this thread)
PyObject *failed(int rc, const char *name) {
    if (rc != CHADQ_ERR_HIP && rc != CHADQ_ERR_DEVICE) Py_RETURN_NONE;
    return PyObject_CallFunction(g_check, "is", rc, name);
}

// linear(x, weight, out_dtype) -> y, or None
PyObject *linear(PyObject *, PyObject *const *args, Py_ssize_t n_args) {
    HANDLE_TH_ERRORS
    if (n_args != 3) Py_RETURN_NONE;
    PyObject *const qw = args[1];
    const bool int4 = (PyObject *)Py_TYPE(qw) == g_int4;
    if (!int4 && (PyObject *)Py_TYPE(qw) != g_int8) Py_RETURN_NONE;
    if (!THPVariable_CheckExact(args[0])) Py_RETURN_NONE;
    const at::Tensor &xt = THPVariable_Unpack(args[0]);
    if (!xt.is_cuda()) Py_RETURN_NONE;  // (before the device is asked for: there may be none)
    const int dev = c10::hip::current_device();
    const at::ScalarType x_type = xt.scalar_type();
    if (x_type != at::kBFloat16 && (int4 || x_type != at::kFloat)) Py_RETURN_NONE;
    const at::Tensor *const x = plain(args[0], x_type, 2, dev);
    if (!x) Py_RETURN_NONE;
    const Ref wo(PyObject_GetAttr(qw, int4 ? s_packed : s_w)), so(PyObject_GetAttr(qw, s_scale));
    const at::Tensor *const w = plain(wo.p, int4 ? at::kByte : at::kChar, 2, dev);
    const at::Tensor *const s = plain(so.p, int4 ? at::kHalf : at::kFloat, int4 ? 2 : 1, dev);
    if (!w || !s) Py_RETURN_NONE;
    const int64_t m = x->size(0), n = w->size(0), k = int4 ? w->size(1) * 2 : w->size(1);
    if (m < 1 || m > INT_MAX || n < 1 || n > INT_MAX || k < 1 || k > INT_MAX || x->size(1) != k || s->size(0) != n || (int4 && s->size(1) * 32 != k))
        Py_RETURN_NONE;
    const bool gemv = m <= kGemvRows && (int4 || x_type == at::kFloat);
    if (!gemv && x_type != at::kBFloat16) Py_RETURN_NONE;
    at::ScalarType y_type = gemv ? at::kFloat : at::kBFloat16;
    if (args[2] != Py_None) {
        if (!THPDtype_Check(args[2])) Py_RETURN_NONE;
        const at::ScalarType want = reinterpret_cast<THPDtype *>(args[2])->scalar_type;
        if (want != y_type && want != at::kBFloat16) Py_RETURN_NONE;
        y_type = want;
    }
    const Entry e = !gemv ? (int4 ? GEMM_I4 : GEMM_I8) : y_type == at::kFloat ? (int4 ? GEMV_I4 : GEMV_I8) : (int4 ? GEMV_I4_BF16 : GEMV_I8_BF16);
    const at::Tensor keep[3] = {*x, *w, *s};  // whatever another thread does with the objects
    const product_fn fn = reinterpret_cast<product_fn>(g_entry[e]);
    // scratch for the K parts of a product that would leave most of the GPU idle; 0: one part is the quicker form
    const size_t need = reinterpret_cast<product_bytes_fn>(g_entry[gemv ? GEMV_BYTES : GEMM_BYTES])((int)m, (int)n, (int)k, !int4);
    at::Tensor y, ws;
    int rc;
    {
        const WithoutLock free;
        if (need) ws = at::empty({(int64_t)need}, keep[0].options().dtype(at::kByte).requires_grad(false));
        y = at::empty({m, n}, keep[0].options().dtype(y_type).requires_grad(false));
        if (!y.unsafeGetTensorImpl()->has_storage() || (need && !ws.unsafeGetTensorImpl()->has_storage())) rc = CHADQ_ERR_NULL;
        else if (need && gemv)
            rc = reinterpret_cast<decode_ws_fn>(g_entry[int4 ? GEMV_I4_WS : GEMV_I8_WS])(
                keep[0].const_data_ptr(), keep[1].const_data_ptr(), keep[2].const_data_ptr(), y.mutable_data_ptr(), (int)m, (int)n, (int)k,
                y_type == at::kBFloat16, ws.mutable_data_ptr(), need, c10::hip::getCurrentHIPStream((c10::DeviceIndex)dev).stream());
        else if (need)
            rc = reinterpret_cast<product_ws_fn>(g_entry[int4 ? GEMM_I4_WS : GEMM_I8_WS])(
                keep[0].const_data_ptr(), keep[1].const_data_ptr(), keep[2].const_data_ptr(), y.mutable_data_ptr(), (int)m, (int)n, (int)k,
                ws.mutable_data_ptr(), need, c10::hip::getCurrentHIPStream((c10::DeviceIndex)dev).stream());
        else rc = fn(keep[0].const_data_ptr(), keep[1].const_data_ptr(), keep[2].const_data_ptr(), y.mutable_data_ptr(), (int)m, (int)n, (int)k,
                     c10::hip::getCurrentHIPStream((c10::DeviceIndex)dev).stream());
    }
    if (rc != 0) return failed(rc, kEntryNames[e]);
    return THPVariable_Wrap(std::move(y));
    END_HANDLE_TH_ERRORS
}

// moe_ffn(x, logits, experts, top_k, renorm) -> y, or None
PyObject *moe_ffn(PyObject *, PyObject *const *args, Py_ssize_t n_args) {
    HANDLE_TH_ERRORS
    if (n_args != 5 || !(PyList_CheckExact(args[2]) || PyTuple_CheckExact(args[2])) || !PyLong_CheckExact(args[3])) Py_RETURN_NONE;
    if (!THPVariable_CheckExact(args[0]) || !THPVariable_Unpack(args[0]).is_cuda()) Py_RETURN_NONE;
    const int dev = c10::hip::current_device();
    const at::Tensor *const x = plain(args[0], at::kBFloat16, 2, dev), *const z = plain(args[1], at::kFloat, 2, dev);
    const Py_ssize_t e = PySequence_Fast_GET_SIZE(args[2]);
    const long top_k = PyLong_AsLong(args[3]);
    if (top_k == -1 && PyErr_Occurred()) PyErr_Clear();
    // (other objects than True, False and ints go through Python's int())
    if (!PyBool_Check(args[4]) && !PyLong_CheckExact(args[4])) Py_RETURN_NONE;
    int overflow = 0;
    const long renorm_value = PyLong_AsLongAndOverflow(args[4], &overflow);
    if (overflow || renorm_value < INT_MIN || renorm_value > INT_MAX) Py_RETURN_NONE;
    const int renorm = (int)renorm_value;
    if (!x || !z || e < 1 || e > kMaxExperts || top_k < 1 || top_k > e) Py_RETURN_NONE;
    const int64_t t = x->size(0), h = x->size(1);
    if (t < 1 || t > INT_MAX || h < 1 || h > INT_MAX || z->size(0) != t || z->size(1) != e) Py_RETURN_NONE;
    chadq_moe_expert_i4g32 arr[kMaxExperts];
    at::Tensor keep[kMaxExperts][6];  // alive until the call is launched
    PyObject *kind = nullptr;
    int64_t f = 0;
    for (Py_ssize_t i = 0; i < e; ++i) {
        PyObject *const triple = PySequence_Fast_GET_ITEM(args[2], i);
        if (!(PyTuple_CheckExact(triple) || PyList_CheckExact(triple)) || PySequence_Fast_GET_SIZE(triple) != 3) Py_RETURN_NONE;
        const void *p[6];
        for (int j = 0; j < 3; ++j) {  // gate, up [F,H], down [H,F]
            PyObject *const m = PySequence_Fast_GET_ITEM(triple, j);
            if (!kind) kind = (PyObject *)Py_TYPE(m);
            if ((PyObject *)Py_TYPE(m) != kind || (kind != g_int4 && kind != g_tiles)) Py_RETURN_NONE;
            const Ref wo(PyObject_GetAttr(m, s_packed)), so(PyObject_GetAttr(m, s_scale));
            const at::Tensor *const w = plain(wo.p, at::kByte, 2, dev), *const s = plain(so.p, at::kHalf, 2, dev);
            if (!w || !s) Py_RETURN_NONE;
            if (i == 0 && j == 0) f = w->size(0);
            const int64_t n = j < 2 ? f : h, k = j < 2 ? h : f;
            if (w->size(0) != n || w->size(1) * 2 != k || s->size(0) != n || s->size(1) * 32 != k) Py_RETURN_NONE;
            keep[i][2 * j] = *w;
            keep[i][2 * j + 1] = *s;
            p[2 * j] = w->const_data_ptr();
            p[2 * j + 1] = s->const_data_ptr();
        }
        arr[i] = chadq_moe_expert_i4g32{};
        memcpy(&arr[i], p, sizeof(p));
    }
    static_assert(sizeof(chadq_moe_expert_i4g32) == 6 * sizeof(void *), "six pointers: gate, up and down with their scales");
    if (f < 1 || f > INT_MAX) Py_RETURN_NONE;
    const size_t need = reinterpret_cast<moe_bytes_fn>(g_entry[MOE_BYTES])((int)t, (int)h, (int)f, (int)e, (int)top_k);
    if (need == 0) Py_RETURN_NONE;
    const Entry entry = kind == g_tiles ? MOE_TILES : MOE_ROWS;
    const moe_fn fn = reinterpret_cast<moe_fn>(g_entry[entry]);
    const at::Tensor xk = *x, zk = *z;  // as keep
    at::Tensor ws, y;
    int rc;
    {
        const WithoutLock free;
        ws = at::empty({(int64_t)need}, xk.options().dtype(at::kByte).requires_grad(false));
        y = at::empty({t, h}, xk.options().requires_grad(false));
        if (!ws.unsafeGetTensorImpl()->has_storage() || !y.unsafeGetTensorImpl()->has_storage()) rc = CHADQ_ERR_NULL;
        else rc = fn(xk.const_data_ptr(), zk.const_data_ptr(), arr, y.mutable_data_ptr(), (int)t, (int)h, (int)f, (int)e, (int)top_k, renorm,
                     ws.mutable_data_ptr(), need, c10::hip::getCurrentHIPStream((c10::DeviceIndex)dev).stream());
    }
    if (rc != 0) return failed(rc, kEntryNames[entry]);
    return THPVariable_Wrap(std::move(y));
    END_HANDLE_TH_ERRORS
}

// gemv_bytes, gemm_bytes(M, N, K, int8 weights) -> scratch bytes of the library's function of that name, for calls that ops.py makes itself: 0.1 us where
// ctypes takes 0.6 to 1.3 to bring home a 0
template <Entry E>
PyObject *bytes_of(PyObject *, PyObject *const *args, Py_ssize_t n_args) {
    int v[4];
    if (n_args != 4) {
        PyErr_SetString(PyExc_TypeError, "M, N, K and whether the weights are int8");
        return nullptr;
    }
    for (int i = 0; i < 4; ++i) {
        const long l = PyLong_AsLong(args[i]);
        if (l == -1 && PyErr_Occurred()) return nullptr;
        if (l < INT_MIN || l > INT_MAX) return PyLong_FromLong(0);  // (what the product itself refuses)
        v[i] = (int)l;
    }
    return PyLong_FromSize_t(reinterpret_cast<product_bytes_fn>(g_entry[E])(v[0], v[1], v[2], v[3]));
}

// bind(addresses of the entry points in the order of Entry, (QWeightInt4G32, QWeightInt8, QWeightInt4G32Tiles), check)
PyObject *bind(PyObject *, PyObject *args) {
    PyObject *addr, *kinds, *check;
    if (!PyArg_ParseTuple(args, "O!O!O", &PyTuple_Type, &addr, &PyTuple_Type, &kinds, &check)) return nullptr;
    if (PyTuple_GET_SIZE(addr) != ENTRIES || PyTuple_GET_SIZE(kinds) != 3 || !PyCallable_Check(check)) {
        PyErr_SetString(PyExc_ValueError, "bind: one address per entry point, three containers and a function");
        return nullptr;
    }
    void *fresh[ENTRIES];
    for (int i = 0; i < ENTRIES; ++i) {
        fresh[i] = PyLong_AsVoidPtr(PyTuple_GET_ITEM(addr, i));
        if (!fresh[i]) {
            if (!PyErr_Occurred()) PyErr_SetString(PyExc_ValueError, "bind: null address");
            return nullptr;
        }
    }
    memcpy(g_entry, fresh, sizeof(fresh));
    PyObject **const slot[3] = {&g_int4, &g_int8, &g_tiles};
    for (int i = 0; i < 3; ++i) {
        PyObject *const k = PyTuple_GET_ITEM(kinds, i);
        Py_INCREF(k);
        Py_XSETREF(*slot[i], k);
    }
    Py_INCREF(check);
    Py_XSETREF(g_check, check);
    Py_RETURN_NONE;
}

PyMethodDef methods[] = {{"linear", (PyCFunction)(void (*)(void))linear, METH_FASTCALL, "linear(x, weight, out_dtype) -> y, or None where the Python path has to look"},
                         {"moe_ffn", (PyCFunction)(void (*)(void))moe_ffn, METH_FASTCALL, "moe_ffn(x, logits, experts, top_k, renorm) -> y, or None"},
                         {"gemv_bytes", (PyCFunction)(void (*)(void))bytes_of<GEMV_BYTES>, METH_FASTCALL, "gemv_bytes(M, N, K, int8) -> bytes"},
                         {"gemm_bytes", (PyCFunction)(void (*)(void))bytes_of<GEMM_BYTES>, METH_FASTCALL, "gemm_bytes(M, N, K, int8) -> bytes"},
                         {"bind", bind, METH_VARARGS, "bind(addresses, containers, check)"},
                         {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_host_call", nullptr, -1, methods};

}  // namespace

PyMODINIT_FUNC PyInit__host_call(void) {
    s_packed = PyUnicode_InternFromString("packed");
    s_scale = PyUnicode_InternFromString("scale");
    s_w = PyUnicode_InternFromString("w");
    if (!s_packed || !s_scale || !s_w) return nullptr;
    return PyModule_Create(&module);
}
