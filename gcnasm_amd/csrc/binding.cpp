// The host's part of the public functions of api.py on ordinary tensors: outputs allocated, the argument block filled from sizes and strides, the
// library called on the current stream.  What an enqueued call of a small layer costs is this and the launch (bound: the host; 1 x 4096 x 4096 with its
// quantiser takes 7.5 us of device time).  us enqueued, api.py's own statements of the same steps over ctypes -> here: that pass, two calls, 17.7 -> 9.1;
// a block-scale GEMM 9.1 -> 4.2; both conversions 14.2 -> 9.1.
//
// Every function returns None for anything but the plain case -- exact torch tensors in ordinary strided GPU memory, Python ints, no dispatch or
// function mode active, shapes and scales that belong together -- and api.py then goes through the checks that name what is wrong, or
// serves the tensor subclass or the mode.  An int is the status of a call that the library refused.
#include <Python.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include <ATen/PythonTorchFunctionTLS.h>
#include <ATen/core/Tensor.h>
#include <ATen/ops/empty.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <c10/hip/HIPFunctions.h>
#include <c10/hip/HIPStream.h>

#include <climits>

#include "../../include/mi355_a8w8.h"

namespace {

// the library's entry points, in the order of api.py's list (addresses: the library that api.py has loaded, whichever build it is)
enum Op { GEMM, GEMM_BLOCKSCALE, FLATMM, GEMM_A16W16, FLATMM_A16W16, GEMM_A4W4, FLATMM_A4W4, GEMM_OPS };
decltype(&a8w8_gemm) g_gemm[GEMM_OPS];
decltype(&a8w8_quantize_ws) g_quantize;
decltype(&a8w8_quantize_workspace_bytes) g_workspace_bytes;
decltype(&a4w4_quantize_mx) g_quantize_mx;
decltype(&a8w8_cvt_f32_to_e4m3) g_encode;
decltype(&a8w8_cvt_e4m3_to_f32) g_decode;

bool modes_active()
{
    return at::impl::torch_function_mode_enabled() || c10::impl::TorchDispatchModeTLS::any_modes_set();
}

// the tensor behind an exact torch.Tensor (or Parameter) in ordinary GPU memory, else nullptr
const at::Tensor* plain(PyObject* o)
{
    if (!THPVariable_CheckExact(o)) return nullptr;
    const at::Tensor& t = THPVariable_Unpack(o);
    static const c10::DispatchKeySet special({c10::DispatchKey::Python, c10::DispatchKey::PythonTLSSnapshot, c10::DispatchKey::FuncTorchBatched,
                                              c10::DispatchKey::FuncTorchGradWrapper, c10::DispatchKey::Functionalize, c10::DispatchKey::Conjugate,
                                              c10::DispatchKey::Negative, c10::DispatchKey::ZeroTensor});
    if (!t.defined() || !t.is_cuda() || t.layout() != at::kStrided || t.is_nested() || t.is_quantized() || t.key_set().has_any(special) ||
        t.unsafeGetTensorImpl()->has_symbolic_sizes_strides() || !t.has_storage())
        return nullptr;
    return &t;
}

// elements side by side along the last dimension
bool rows_contiguous(const at::Tensor& t) { return t.size(-1) <= 1 || t.stride(-1) == 1; }

// sizes and strides that the C ABI's ints hold
template <class... I>
bool ints(I... v)
{
    return ((v <= INT_MAX) && ...);
}

// fp32 [rows, k] that a quantiser reads row by row (narrower elements would be read past their end)
const at::Tensor* fp32_rows(PyObject* o)
{
    const at::Tensor* x = plain(o);
    return x && x->scalar_type() == at::kFloat && x->dim() == 2 && x->size(0) > 0 && x->size(1) > 0 && rows_contiguous(*x) &&
                   ints(x->size(0), x->size(1), x->stride(0)) ? x : nullptr;
}

bool as_int(PyObject* o, long& v)
{
    if (!PyLong_Check(o)) return false;      // (bools are ints)
    int over = 0;
    v = PyLong_AsLongAndOverflow(o, &over);
    return over == 0;
}

at::Tensor allocate(at::IntArrayRef sizes, at::ScalarType type, const at::Tensor& like)
{
    return at::empty(sizes, at::TensorOptions().dtype(type).device(like.device()));
}

void* stream() { return c10::hip::getCurrentHIPStream().stream(); }

int64_t mx_tiled(int64_t rows, int64_t k) { return (k + 511) / 512 * ((rows + 63) / 64) * 1024; }

PyObject* pair(const at::Tensor& q, const at::Tensor& s)
{
    PyObject* a = THPVariable_Wrap(q);
    PyObject* b = a ? THPVariable_Wrap(s) : nullptr;
    PyObject* t = b ? PyTuple_Pack(2, a, b) : nullptr;
    Py_XDECREF(a);
    Py_XDECREF(b);
    return t;
}

// ------------------------------------------------------------ quantisers: (x, scale_mode, group_rows), (x, tiled) -> (q, scales)
PyObject* quantize(PyObject*, PyObject* const* args, Py_ssize_t count)
{
    HANDLE_TH_ERRORS
    long mode, group;
    const at::Tensor* x = count == 3 && !modes_active() ? fp32_rows(args[0]) : nullptr;
    if (!x || !as_int(args[1], mode) || !as_int(args[2], group)) Py_RETURN_NONE;
    const int64_t rows = x->size(0), k = x->size(1);
    if (mode < A8W8_SCALE_TENSOR || mode > A8W8_SCALE_MX_E8M0_TILED) Py_RETURN_NONE;
    const at::Tensor q = allocate({rows, k}, at::kByte, *x);
    const at::Tensor s = mode == A8W8_SCALE_TENSOR                                ? allocate({1}, at::kFloat, *x)
                         : mode == A8W8_SCALE_ROWCOL                              ? allocate({rows}, at::kFloat, *x)
                         : mode == A8W8_SCALE_BLOCK_1x128_128x128 && group == 1   ? allocate({k / 128, rows}, at::kFloat, *x)
                         : mode == A8W8_SCALE_BLOCK_1x128_128x128                 ? allocate({rows / 128, k / 128}, at::kFloat, *x)
                         : mode == A8W8_SCALE_MX_E8M0_1x32                        ? allocate({rows, k / 32}, at::kByte, *x)
                                                                                  : allocate({mx_tiled(rows, k)}, at::kByte, *x);
    const void* src = x->data_ptr();
    void *qp = q.data_ptr(), *sp = s.data_ptr(), *st = stream();
    const int64_t ld = x->stride(0);
    // (the workspace goes back to the allocator with this call: to be handed out again behind it on the stream that it was allocated on, which is the
    // launches' own only on the current device)
    const size_t ws_bytes = x->device().index() == c10::hip::current_device() ? g_workspace_bytes((int)rows, (int)k, (int)mode) : 0;
    const at::Tensor ws = ws_bytes ? allocate({(int64_t)ws_bytes}, at::kByte, *x) : at::Tensor();
    void* wp = ws_bytes ? ws.data_ptr() : nullptr;
    int status;
    Py_BEGIN_ALLOW_THREADS
    status = g_quantize((const float*)src, (int)rows, (int)k, (int)ld, (uint8_t*)qp, sp, (int)mode, (int)group, wp, ws_bytes, st);
    Py_END_ALLOW_THREADS
    return status ? PyLong_FromLong(status) : pair(q, s);
    END_HANDLE_TH_ERRORS
}

PyObject* quantize_mxfp4(PyObject*, PyObject* const* args, Py_ssize_t count)
{
    HANDLE_TH_ERRORS
    long tiled;
    const at::Tensor* x = count == 2 && !modes_active() ? fp32_rows(args[0]) : nullptr;
    if (!x || !as_int(args[1], tiled)) Py_RETURN_NONE;
    const int64_t rows = x->size(0), k = x->size(1), ld = x->stride(0);
    const at::Tensor q = allocate({rows, k / 2}, at::kByte, *x);
    const at::Tensor s = tiled ? allocate({mx_tiled(rows, k)}, at::kByte, *x) : allocate({rows, k / 32}, at::kByte, *x);
    const void* src = x->data_ptr();
    void *qp = q.data_ptr(), *sp = s.data_ptr(), *st = stream();
    int status;
    Py_BEGIN_ALLOW_THREADS
    status = g_quantize_mx((const float*)src, (int)rows, (int)k, (int)ld, (uint8_t*)qp, (uint8_t*)sp, (int)tiled, st);
    Py_END_ALLOW_THREADS
    return status ? PyLong_FromLong(status) : pair(q, s);
    END_HANDLE_TH_ERRORS
}

// ------------------------------------------------------------ conversions: (x, dialect, clamp240), (codes, dialect) -> out
PyObject* encode(PyObject*, PyObject* const* args, Py_ssize_t count)
{
    HANDLE_TH_ERRORS
    long dialect, clamp;
    const at::Tensor* x = count == 3 && !modes_active() ? plain(args[0]) : nullptr;
    if (!x || x->scalar_type() != at::kFloat || !x->is_contiguous() || !as_int(args[1], dialect) || !as_int(args[2], clamp)) Py_RETURN_NONE;
    const at::Tensor out = allocate(x->sizes(), at::kByte, *x);
    const void* src = x->data_ptr();
    void *dst = out.data_ptr(), *st = stream();
    const size_t n = (size_t)x->numel();
    int status;
    Py_BEGIN_ALLOW_THREADS
    status = g_encode((const float*)src, (uint8_t*)dst, n, (int)dialect, (int)clamp, st);
    Py_END_ALLOW_THREADS
    return status ? PyLong_FromLong(status) : THPVariable_Wrap(out);
    END_HANDLE_TH_ERRORS
}

PyObject* decode(PyObject*, PyObject* const* args, Py_ssize_t count)
{
    HANDLE_TH_ERRORS
    long dialect;
    const at::Tensor* x = count == 2 && !modes_active() ? plain(args[0]) : nullptr;
    if (!x || x->element_size() != 1 || !x->is_contiguous() || !as_int(args[1], dialect)) Py_RETURN_NONE;
    const at::Tensor out = allocate(x->sizes(), at::kFloat, *x);
    const void* src = x->data_ptr();
    void *dst = out.data_ptr(), *st = stream();
    const size_t n = (size_t)x->numel();
    int status;
    Py_BEGIN_ALLOW_THREADS
    status = g_decode((const uint8_t*)src, (float*)dst, n, (int)dialect, st);
    Py_END_ALLOW_THREADS
    return status ? PyLong_FromLong(status) : THPVariable_Wrap(out);
    END_HANDLE_TH_ERRORS
}

// ------------------------------------------------------------ GEMMs: (op, a, b, sfa, sfb, scale_mode, c, c_dtype, n) -> c

// elements of one batch entry's scale array (scale_elements of api.py)
int64_t scale_elements(long mode, int64_t rows, int64_t k, bool weight_side)
{
    switch (mode) {
        case A8W8_SCALE_TENSOR: return 1;
        case A8W8_SCALE_ROWCOL: return rows;
        case A8W8_SCALE_BLOCK_1x128_128x128: return (weight_side ? (rows + 127) / 128 : rows) * (k / 128);
        case A8W8_SCALE_MX_E8M0_1x32: return rows * (k / 32);
        default: return mx_tiled(rows, k);
    }
}

// a one-byte array of a contiguous tensor, as many elements as the kernels read
bool fp4_scales_ok(const at::Tensor& t, int64_t need) { return t.is_contiguous() && t.element_size() == 1 && t.numel() >= need; }

PyObject* gemm(PyObject*, PyObject* const* args, Py_ssize_t count)
{
    HANDLE_TH_ERRORS
    long op, mode, c_dtype, n_given = 0;
    if (count != 9 || modes_active() || !as_int(args[0], op) || op < 0 || op >= GEMM_OPS || !as_int(args[5], mode) || !as_int(args[7], c_dtype)) Py_RETURN_NONE;
    const bool shuffled = args[8] != Py_None;
    if (shuffled && !as_int(args[8], n_given)) Py_RETURN_NONE;
    const at::Tensor *a = plain(args[1]), *b = plain(args[2]), *sfa = plain(args[3]), *sfb = plain(args[4]);
    if (!a || !b || !sfa || !sfb || mode < A8W8_SCALE_TENSOR || mode > A8W8_SCALE_MX_E8M0_TILED || (c_dtype != A8W8_C_BF16 && c_dtype != A8W8_C_FP32)) Py_RETURN_NONE;
    const bool fp4 = op == GEMM_A4W4 || op == FLATMM_A4W4, scaled = op != GEMM_A16W16 && op != FLATMM_A16W16;
    const bool batched = a->dim() == 3;
    if ((a->dim() != 2 && !batched) || (fp4 && batched) || !(shuffled ? b->dim() == 1 || b->dim() == 2 : b->dim() == 2 || (b->dim() == 3 && batched)))
        Py_RETURN_NONE;
    const int64_t element_bytes = scaled ? 1 : 2;
    if (!rows_contiguous(*a) || (int64_t)a->element_size() != element_bytes) Py_RETURN_NONE;
    if (!shuffled && (!rows_contiguous(*b) || (int64_t)b->element_size() != element_bytes || b->size(-1) < a->size(-1))) Py_RETURN_NONE;
    if (shuffled && (!b->is_contiguous() || (int64_t)b->nbytes() < n_given * a->size(-1) * element_bytes)) Py_RETURN_NONE;
    const int64_t per_byte = fp4 ? 2 : 1, batch = batched ? a->size(0) : 1, m = a->size(-2), k = a->size(-1) * per_byte, n = shuffled ? n_given : b->size(-2);
    if (batch <= 0 || m <= 0 || n <= 0 || k <= 0) Py_RETURN_NONE;

    const int64_t stride_b = shuffled ? k : b->stride(-2) * per_byte;
    int64_t a_batch = m * a->stride(-2) * per_byte, b_batch = n * stride_b;
    int64_t sfa_batch = scale_elements(mode, m, k, false), sfb_batch = scale_elements(mode, n, k, true);
    if (mode == A8W8_SCALE_BLOCK_1x128_128x128) sfb_batch = n / 128 * (k / 128);
    if (batched) {
        a_batch = a->stride(0);
        if (shuffled) {
            const int64_t per_entry = n * k * (int64_t)a->element_size() / (int64_t)b->element_size();
            if (b->numel() == batch * per_entry) b_batch = n * k;
            else if (b->numel() == per_entry) b_batch = sfb_batch = 0;
            else Py_RETURN_NONE;
        } else if (b->dim() == 3) {
            if (b->size(0) != batch) Py_RETURN_NONE;
            b_batch = b->stride(0);
        } else {
            b_batch = sfb_batch = 0;      // one weight matrix, and one set of weight scales, for every batch entry
        }
    }
    if (fp4 && (mode < A8W8_SCALE_MX_E8M0_1x32 || !fp4_scales_ok(*sfa, sfa_batch) || !fp4_scales_ok(*sfb, sfb_batch))) Py_RETURN_NONE;
    if (scaled && !fp4) {
        const at::ScalarType want = mode >= A8W8_SCALE_MX_E8M0_1x32 ? at::kByte : at::kFloat;
        if (!sfa->is_contiguous() || !sfb->is_contiguous() || sfa->scalar_type() != want || sfb->scalar_type() != want) Py_RETURN_NONE;
        const bool shared = batch > 1 && b_batch == 0;
        const int64_t per_b = scale_elements(mode, n, k, true), has_b = sfb->numel();
        if (sfa->numel() < batch * scale_elements(mode, m, k, false) || has_b < (shared ? per_b : batch * per_b) || (shared && has_b >= batch * per_b && has_b > per_b))
            Py_RETURN_NONE;
    }

    at::Tensor out;
    const at::Tensor* c = nullptr;
    if (args[6] == Py_None) {
        const at::ScalarType type = c_dtype == A8W8_C_BF16 ? at::kBFloat16 : at::kFloat;
        out = batched ? allocate({batch, m, n}, type, *a) : allocate({m, n}, type, *a);
        c = &out;
    } else {
        c = plain(args[6]);
        if (!c || (c->scalar_type() != at::kBFloat16 && c->scalar_type() != at::kFloat) || c->dim() != a->dim() || (batched && c->size(0) != batch) || c->size(-2) != m ||
            c->size(-1) != n || (n > 1 && c->stride(-1) != 1))
            Py_RETURN_NONE;
        c_dtype = c->scalar_type() == at::kBFloat16 ? A8W8_C_BF16 : A8W8_C_FP32;
    }
    if (!ints(m, n, k, batch, a->stride(-2) * per_byte, stride_b, c->stride(-2)) || (batch > 1 && !ints(a_batch, b_batch, c->stride(0), sfa_batch, sfb_batch))) Py_RETURN_NONE;
    a8w8_gemm_args g;
    g.a = a->data_ptr(); g.b = b->data_ptr(); g.c = c->data_ptr();
    g.m = (int)m; g.n = (int)n; g.k = (int)k; g.batch = (int)batch;
    g.stride_a = (int)(a->stride(-2) * per_byte); g.stride_b = (int)stride_b; g.stride_c = (int)c->stride(-2);
    g.stride_a_batch = (int)a_batch; g.stride_b_batch = (int)b_batch; g.stride_c_batch = (int)(batched ? c->stride(0) : m * c->stride(-2));
    g.sfa = sfa->data_ptr(); g.sfb = sfb->data_ptr();
    g.stride_sfa = mode == A8W8_SCALE_BLOCK_1x128_128x128 ? (int)m : mode == A8W8_SCALE_MX_E8M0_1x32 ? (int)(k / 32) : 0;
    g.stride_sfb = mode == A8W8_SCALE_ROWCOL ? 1 : mode == A8W8_SCALE_BLOCK_1x128_128x128 ? (int)(k / 128) : mode == A8W8_SCALE_MX_E8M0_1x32 ? (int)(k / 32) : 0;
    g.stride_sfa_batch = (int)sfa_batch; g.stride_sfb_batch = (int)sfb_batch;
    g.scale_mode = (int)mode; g.c_dtype = (int)c_dtype; g.b_preshuffled = shuffled;
    void* st = stream();
    int status;
    Py_BEGIN_ALLOW_THREADS
    status = g_gemm[op](&g, st);
    Py_END_ALLOW_THREADS
    if (status) return PyLong_FromLong(status);
    if (args[6] == Py_None) return THPVariable_Wrap(out);
    Py_INCREF(args[6]);
    return args[6];
    END_HANDLE_TH_ERRORS
}

// (address, ...) of the entry points, in the order of their variables above
PyObject* connect(PyObject*, PyObject* const* args, Py_ssize_t count)
{
    void* p[GEMM_OPS + 5];
    if (count != GEMM_OPS + 5) {
        PyErr_SetString(PyExc_TypeError, "one address per entry point");
        return nullptr;
    }
    for (Py_ssize_t i = 0; i < count; ++i) {
        p[i] = PyLong_AsVoidPtr(args[i]);
        if (!p[i]) {
            if (!PyErr_Occurred()) PyErr_SetString(PyExc_ValueError, "null entry point");
            return nullptr;
        }
    }
    for (int i = 0; i < GEMM_OPS; ++i) g_gemm[i] = (decltype(&a8w8_gemm))p[i];
    g_quantize = (decltype(&a8w8_quantize_ws))p[GEMM_OPS];
    g_quantize_mx = (decltype(&a4w4_quantize_mx))p[GEMM_OPS + 1];
    g_encode = (decltype(&a8w8_cvt_f32_to_e4m3))p[GEMM_OPS + 2];
    g_decode = (decltype(&a8w8_cvt_e4m3_to_f32))p[GEMM_OPS + 3];
    g_workspace_bytes = (decltype(&a8w8_quantize_workspace_bytes))p[GEMM_OPS + 4];
    Py_RETURN_NONE;
}

#define FASTCALL(f) (PyCFunction)(void (*)(void)) f, METH_FASTCALL
PyMethodDef methods[] = {{"connect", FASTCALL(connect), nullptr}, {"quantize", FASTCALL(quantize), nullptr}, {"quantize_mxfp4", FASTCALL(quantize_mxfp4), nullptr},
                         {"encode", FASTCALL(encode), nullptr},   {"decode", FASTCALL(decode), nullptr},     {"gemm", FASTCALL(gemm), nullptr},
                         {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_binding", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

// torch_build: the torch whose headers these are (api.py compares it with the torch that is loaded)
PyMODINIT_FUNC PyInit__binding(void)
{
    PyObject* m = PyModule_Create(&module);
    if (m && PyModule_AddStringConstant(m, "torch_build", A8W8_TORCH_BUILD) != 0) Py_CLEAR(m);
    return m;
}
