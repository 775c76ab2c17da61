// Native side of the calls that a program makes most often: argument checks, output allocation and the call into libmase_hip.so in one
// step from Python.  A small cast takes 3 us on the GPU and as long to launch; through ctypes and Python wrappers it took 8 - 13 us of
// host time, now 4.5 - 6.
//
// Every function takes the call only where it is plain: exact torch tensors on the current GPU, contiguous, 16-byte aligned, of
// a type that the kernels read, no dispatch or function mode active.  Anything else (and any error that the library reports) returns
// None, and the Python wrapper does what it always did: it copies, converts, switches the device, or raises the error.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <ATen/core/Tensor.h>
#include <ATen/PythonTorchFunctionTLS.h>
#include <ATen/autocast_mode.h>
#include <ATen/core/grad_mode.h>
#include <ATen/ops/empty.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <c10/core/impl/VirtualGuardImpl.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/jit/frontend/tracer.h>

#include "../../../include/mase_hip.h"
#include "../../../include/mase_hip_scores.h"
#include "../../../include/mase_hip_linear.h"

namespace {

PyObject* g_raw_stream = nullptr;   // torch._C._cuda_getCurrentRawStream

int dtype_code(at::ScalarType t) {
    return t == at::kFloat ? 0 : t == at::kHalf ? 1 : t == at::kBFloat16 ? 2 : -1;
}
const at::ScalarType kDtypes[3] = {at::kFloat, at::kHalf, at::kBFloat16};

// an exact tensor on a GPU that owns its data as it lies
const at::Tensor* gpu_tensor(PyObject* o) {
    if (!THPVariable_CheckExact(o)) return nullptr;
    const at::Tensor& t = THPVariable_Unpack(o);
    if (!t.defined() || !t.is_cuda() || t.layout() != at::kStrided || !t.unsafeGetTensorImpl()->has_storage() || t.is_neg() || t._is_zerotensor()) return nullptr;
    return &t;
}
bool dense(const at::Tensor& t) { return t.is_contiguous() && reinterpret_cast<uintptr_t>(t.data_ptr()) % 16 == 0; }

// stream of the current device if `t` is on it and nothing wants to see the calls; false: not a plain call
bool stream_of(const at::Tensor& t, void** stream) {
    static const c10::impl::VirtualGuardImpl guard(c10::DeviceType::CUDA);
    if (c10::impl::TorchDispatchModeTLS::any_modes_set() || at::impl::PythonTorchFunctionTLS::stack_len() > 0) return false;
    const auto device = t.device().index();
    if (guard.getDevice().index() != device) return false;
    PyObject* const index = PyLong_FromLong(device);
    if (!index) return PyErr_Clear(), false;
    PyObject* const raw = PyObject_CallOneArg(g_raw_stream, index);
    Py_DECREF(index);
    if (!raw) return PyErr_Clear(), false;
    *stream = PyLong_AsVoidPtr(raw);
    Py_DECREF(raw);
    if (PyErr_Occurred()) return PyErr_Clear(), false;
    return true;
}

// the whole number that `o` stands for; false: none that a long holds (a block axis of 1.0 is for the wrappers to refuse)
bool whole(PyObject* o, long& v) {
    v = PyLong_AsLong(o);
    if (v == -1 && PyErr_Occurred()) return PyErr_Clear(), false;
    return true;
}

// (block_size, exp_bits, frac_bits, finite, round mode or -1) of MXFP formats, (exp_bits, frac_bits, finite, round mode) of minifloat ones
template <int N>
bool ints(PyObject* tuple, long (&v)[N]) {
    if (!PyTuple_CheckExact(tuple) || PyTuple_GET_SIZE(tuple) != N) return false;
    for (int i = 0; i < N; ++i)
        if (!whole(PyTuple_GET_ITEM(tuple, i), v[i])) return false;
    return v[N - 1] >= 0;
}
// code of the output type: None (that of `t`) or a code
int out_code(PyObject* o, const at::Tensor& t) {
    if (o == Py_None) return dtype_code(t.scalar_type());
    long c;
    return whole(o, c) && c >= 0 && c < 3 ? (int)c : -1;
}

using Sizes = c10::SmallVector<int64_t, 6>;
Sizes sizes_of(const at::Tensor& t) { return Sizes(t.sizes().begin(), t.sizes().end()); }

// blocks along axis `dim` of a contiguous tensor: [outer, k, inner]; false: not an axis
bool extents(const at::Tensor& t, long dim, int64_t& outer, int64_t& k, int64_t& inner) {
    const int64_t nd = t.dim();
    if (dim < -nd || dim >= nd) return false;
    if (dim < 0) dim += nd;
    outer = inner = 1;
    for (int64_t i = 0; i < dim; ++i) outer *= t.size(i);
    for (int64_t i = dim + 1; i < nd; ++i) inner *= t.size(i);
    k = t.size(dim);
    return dim == nd - 1 || k % 32 == 0;
}

at::Tensor empty(at::IntArrayRef sizes, at::ScalarType dtype, at::Device device) { return at::empty(sizes, at::TensorOptions().dtype(dtype).device(device)); }

// Other Python threads run while one allocates (which can wait for the GPU) and launches (which waits where the queue is full), as they do
// beside torch's own calls.  What such a thread could change (sizes, data) is read before; nothing of Python's is touched in its scope.
struct WithoutGil {
    PyThreadState* const state = PyEval_SaveThread();
    WithoutGil() = default;
    WithoutGil(const WithoutGil&) = delete;
    ~WithoutGil() { PyEval_RestoreThread(state); }
};

#define PLAIN(cond) \
    if (!(cond)) Py_RETURN_NONE

// extract_mxfp(x, block_dim, format) -> (scales [n / B, 1], elements [n / B, B])
PyObject* extract_mxfp(PyObject*, PyObject* const* a, Py_ssize_t n_args) {
    HANDLE_TH_ERRORS
    PLAIN(n_args == 3);
    const at::Tensor* const x = gpu_tensor(a[0]);
    long f[5], dim;
    PLAIN(x && dense(*x) && ints(a[2], f) && whole(a[1], dim));
    int64_t outer, k, inner;
    void* stream;
    const int dt = dtype_code(x->scalar_type());
    const int64_t n = x->numel(), B = f[0];
    PLAIN(dt >= 0 && n > 0 && B > 0 && n % B == 0 && extents(*x, dim, outer, k, inner) && stream_of(*x, &stream));
    const bool last = dim == -1 || dim == x->dim() - 1;
    PLAIN(last || B == 32);
    const void* const data = x->data_ptr();
    const at::Device device = x->device();
    at::Tensor scales, elements;
    int rc;
    {
        const WithoutGil released;
        scales = empty({n / B, 1}, at::kByte, device);
        elements = empty({n / B, B}, at::kByte, device);
        rc = last ? mase_hip_extract_mxfp(data, dt, scales.data_ptr<uint8_t>(), elements.data_ptr<uint8_t>(), n, (int)B, (int)f[1], (int)f[2], (int)f[3], (int)f[4], stream)
                  : mase_hip_extract_mxfp_strided(data, dt, scales.data_ptr<uint8_t>(), elements.data_ptr<uint8_t>(), outer, k, inner, 32, (int)f[1], (int)f[2], (int)f[3], (int)f[4],
                                                  stream);
    }
    PLAIN(rc == 0);
    PyObject* const s = THPVariable_Wrap(std::move(scales));
    PyObject* const e = s ? THPVariable_Wrap(std::move(elements)) : nullptr;
    PyObject* const r = e ? PyTuple_New(2) : nullptr;
    if (!r) {
        Py_XDECREF(s);
        Py_XDECREF(e);
        return nullptr;
    }
    PyTuple_SET_ITEM(r, 0, s);
    PyTuple_SET_ITEM(r, 1, e);
    return r;
    END_HANDLE_TH_ERRORS
}

// qdq_mxfp(x, block_dim, format, output code or None) -> tensor of x's shape
PyObject* qdq_mxfp(PyObject*, PyObject* const* a, Py_ssize_t n_args) {
    HANDLE_TH_ERRORS
    PLAIN(n_args == 4);
    const at::Tensor* const x = gpu_tensor(a[0]);
    long f[5], dim;
    PLAIN(x && dense(*x) && ints(a[2], f) && whole(a[1], dim));
    int64_t outer, k, inner;
    void* stream;
    const int dt = dtype_code(x->scalar_type()), od = out_code(a[3], *x);
    const int64_t n = x->numel(), B = f[0];
    PLAIN(dt >= 0 && od >= 0 && n > 0 && B > 0 && n % B == 0 && extents(*x, dim, outer, k, inner) && stream_of(*x, &stream));
    const bool last = dim == -1 || dim == x->dim() - 1;
    PLAIN(last || B == 32);
    const Sizes sizes = sizes_of(*x);
    const void* const data = x->data_ptr();
    const at::Device device = x->device();
    at::Tensor out;
    int rc;
    {
        const WithoutGil released;
        out = empty(sizes, kDtypes[od], device);
        rc = last ? mase_hip_qdq_mxfp(data, dt, out.data_ptr(), od, n, (int)B, (int)f[1], (int)f[2], (int)f[3], (int)f[4], stream)
                  : mase_hip_qdq_mxfp_strided(data, dt, out.data_ptr(), od, outer, k, inner, 32, (int)f[1], (int)f[2], (int)f[3], (int)f[4], stream);
    }
    PLAIN(rc == 0);
    return THPVariable_Wrap(std::move(out));
    END_HANDLE_TH_ERRORS
}

// compose_mxfp(scales, elements, format, output code, shape of the tensor with its block axis last) -> tensor of that shape
PyObject* compose_mxfp(PyObject*, PyObject* const* a, Py_ssize_t n_args) {
    HANDLE_TH_ERRORS
    PLAIN(n_args == 5);
    const at::Tensor *const scales = gpu_tensor(a[0]), *const elements = gpu_tensor(a[1]);
    long f[5];
    PLAIN(scales && elements && dense(*scales) && dense(*elements) && ints(a[2], f) && PyTuple_Check(a[4]));
    const int od = out_code(a[3], *elements);
    const int64_t n = elements->numel(), B = f[0];
    PLAIN(od >= 0 && n > 0 && B > 0 && n % B == 0 && scales->numel() == n / B && scales->scalar_type() == at::kByte && elements->scalar_type() == at::kByte &&
          scales->device() == elements->device());
    Sizes shape;
    int64_t total = 1;
    for (Py_ssize_t i = 0; i < PyTuple_GET_SIZE(a[4]); ++i) {
        long d;
        PLAIN(whole(PyTuple_GET_ITEM(a[4], i), d) && d > 0);
        shape.push_back(d);
        PLAIN(!__builtin_mul_overflow(total, (int64_t)d, &total));
    }
    void* stream;
    PLAIN(total == n && stream_of(*elements, &stream));
    const uint8_t *const scale_data = scales->data_ptr<uint8_t>(), *const element_data = elements->data_ptr<uint8_t>();
    const at::Device device = elements->device();
    at::Tensor out;
    int rc;
    {
        const WithoutGil released;
        out = empty(shape, kDtypes[od], device);
        rc = mase_hip_compose_mxfp(scale_data, element_data, out.data_ptr(), od, n, (int)B, (int)f[1], (int)f[2], (int)f[3], stream);
    }
    PLAIN(rc == 0);
    return THPVariable_Wrap(std::move(out));
    END_HANDLE_TH_ERRORS
}

// minifloat(kind, x, format, output code or None): kind 0 extract (uint16 codes), 1 compose (x: codes), 2 quantise-dequantise
PyObject* minifloat(PyObject*, PyObject* const* a, Py_ssize_t n_args) {
    HANDLE_TH_ERRORS
    PLAIN(n_args == 4);
    const at::Tensor* const x = gpu_tensor(a[1]);
    long kind, f[4];
    PLAIN(whole(a[0], kind) && x && dense(*x) && ints(a[2], f));
    const int dt = dtype_code(x->scalar_type()), od = kind == 0 ? 0 : out_code(a[3], *x);
    const int64_t n = x->numel();
    void* stream;
    PLAIN(kind >= 0 && kind <= 2 && n > 0 && od >= 0 && (kind == 1 ? x->scalar_type() == at::kUInt16 : dt >= 0) && stream_of(*x, &stream));
    const Sizes sizes = sizes_of(*x);
    const void* const data = x->data_ptr();
    const at::Device device = x->device();
    const int E = (int)f[0], M = (int)f[1], fin = (int)f[2], rm = (int)f[3];
    at::Tensor out;
    int rc;
    {
        const WithoutGil released;
        out = empty(sizes, kind == 0 ? at::kUInt16 : kDtypes[od], device);
        rc = kind == 0   ? mase_hip_extract_minifloat(data, dt, static_cast<uint16_t*>(out.data_ptr()), n, E, M, fin, rm, stream)
             : kind == 1 ? mase_hip_compose_minifloat(static_cast<const uint16_t*>(data), out.data_ptr(), od, n, E, M, fin, stream)
                         : mase_hip_qdq_minifloat(data, dt, out.data_ptr(), od, n, E, M, fin, rm, stream);
    }
    PLAIN(rc == 0);
    return THPVariable_Wrap(std::move(out));
    END_HANDLE_TH_ERRORS
}

// what the linears have in common beside x and W: the bias (a vector of N, or None), the stream, the shape of the outputs
struct LinearRest {
    const void* bias = nullptr;
    int bias_dtype = 0;
    void* stream = nullptr;
    Sizes shape;
};
bool linear_rest(const at::Tensor& x, int64_t N, PyObject* bias, LinearRest& r) {
    if (bias != Py_None) {
        const at::Tensor* const b = THPVariable_Check(bias) ? &THPVariable_Unpack(bias) : nullptr;
        if (!b || !b->is_cuda() || b->device() != x.device() || !b->unsafeGetTensorImpl()->has_storage() || !b->is_contiguous() || b->numel() != N) return false;
        r.bias_dtype = dtype_code(b->scalar_type());
        if (r.bias_dtype < 0) return false;
        r.bias = b->data_ptr();
    }
    r.shape = sizes_of(x);
    r.shape.back() = N;
    return stream_of(x, &r.stream);
}

// linear_scaled(x [.., K] bf16, exp_bits, frac_bits, minifloat, w_codes, w_scales, N, bias or None) -> [.., N]
PyObject* linear_scaled(PyObject*, PyObject* const* a, Py_ssize_t n_args) {
    HANDLE_TH_ERRORS
    PLAIN(n_args == 8);
    const at::Tensor *const x = gpu_tensor(a[0]), *const codes = gpu_tensor(a[4]), *const w_sc = gpu_tensor(a[5]);
    PLAIN(x && codes && w_sc && dense(*x) && x->dim() > 0 && x->scalar_type() == at::kBFloat16 && codes->device() == x->device() && w_sc->device() == x->device());
    PLAIN(codes->is_contiguous() && w_sc->is_contiguous() && codes->scalar_type() == at::kByte && w_sc->scalar_type() == at::kInt && codes->dim() == 2);
    long e, m, mini, N;
    PLAIN(whole(a[1], e) && whole(a[2], m) && whole(a[3], mini) && whole(a[6], N));
    const int64_t K = x->size(-1), M = K > 0 ? x->numel() / K : 0;
    PLAIN(M > 0 && N > 0 && codes->size(1) == K && codes->size(0) >= N && w_sc->numel() >= K / 128 * codes->size(0));
    LinearRest r;
    PLAIN(linear_rest(*x, N, a[7], r));
    const void* const data = x->data_ptr();
    const uint8_t* const code_data = codes->data_ptr<uint8_t>();
    const uint32_t* const scale_data = reinterpret_cast<const uint32_t*>(w_sc->data_ptr<int>());
    const at::Device device = x->device();
    at::Tensor scratch, y;
    int rc = -1;
    {
        const WithoutGil released;
        if (mase_hip_mxfp_linear_few_plan(M, N, K)) {
            y = empty(r.shape, at::kBFloat16, device);
            rc = mase_hip_mxfp_linear_few(data, (int)e, (int)m, (int)mini, code_data, scale_data, r.bias, r.bias_dtype, y.data_ptr(), M, N, K, r.stream);
        } else if (const int64_t bytes = mase_hip_mxfp_linear_scaled_scratch_bytes(M, N, K); bytes > 0) {
            scratch = empty({bytes}, at::kByte, device);
            y = empty(r.shape, at::kBFloat16, device);
            rc = mase_hip_mxfp_linear_scaled(data, 2, (int)e, (int)m, (int)mini, code_data, scale_data, r.bias, r.bias_dtype, y.data_ptr(), 2, M, N, K, scratch.data_ptr(), bytes, r.stream);
        }
    }
    PLAIN(rc == 0);
    return THPVariable_Wrap(std::move(y));
    END_HANDLE_TH_ERRORS
}

// linear_packed(x [.., K] bf16, exp_bits, frac_bits, minifloat, w_codes, w_scales, exp_bits and frac_bits of W, N, bias or None) -> [.., N]
PyObject* linear_packed(PyObject*, PyObject* const* a, Py_ssize_t n_args) {
    HANDLE_TH_ERRORS
    PLAIN(n_args == 10);
    const at::Tensor *const x = gpu_tensor(a[0]), *const codes = gpu_tensor(a[4]), *const w_sc = gpu_tensor(a[5]);
    PLAIN(x && codes && w_sc && dense(*x) && x->dim() > 0 && x->scalar_type() == at::kBFloat16 && codes->device() == x->device() && w_sc->device() == x->device());
    PLAIN(codes->is_contiguous() && w_sc->is_contiguous() && codes->scalar_type() == at::kByte && w_sc->scalar_type() == at::kInt);
    long e, m, mini, we, wm, N;
    PLAIN(whole(a[1], e) && whole(a[2], m) && whole(a[3], mini) && whole(a[6], we) && whole(a[7], wm) && whole(a[8], N));
    const int64_t K = x->size(-1), M = K > 0 ? x->numel() / K : 0;
    PLAIN(M > 0 && N > 0 && K < (1 << 27));
    const int64_t code_bytes = mase_hip_packed_weight_bytes(N, K, (int)we, (int)wm);
    PLAIN(code_bytes > 0 && codes->numel() == code_bytes && w_sc->numel() == K / 128 * ((N + 255) / 256 * 256));
    LinearRest r;
    PLAIN(linear_rest(*x, N, a[9], r));
    const void* const data = x->data_ptr();
    const uint8_t* const code_data = codes->data_ptr<uint8_t>();
    const uint32_t* const scale_data = reinterpret_cast<const uint32_t*>(w_sc->data_ptr<int>());
    const at::Device device = x->device();
    at::Tensor scratch, y;
    int rc = -1;
    {
        const WithoutGil released;
        const int64_t bytes = mase_hip_mxfp_linear_packed_scratch_bytes(M, N, K, (int)we, (int)wm);
        if (bytes > 0) scratch = empty({bytes}, at::kByte, device);
        y = empty(r.shape, at::kBFloat16, device);
        rc = mase_hip_mxfp_linear_packed(data, (int)e, (int)m, (int)mini, code_data, scale_data, (int)we, (int)wm, r.bias, r.bias_dtype, y.data_ptr(), M, N, K,
                                         bytes > 0 ? scratch.data_ptr() : nullptr, bytes, r.stream);
    }
    PLAIN(rc == 0);
    return THPVariable_Wrap(std::move(y));
    END_HANDLE_TH_ERRORS
}

// linear_packed_dense(x [.., K] bf16, w_codes, w_scales, exp_bits and frac_bits of W, N, bias or None) -> [.., N]
PyObject* linear_packed_dense(PyObject*, PyObject* const* a, Py_ssize_t n_args) {
    HANDLE_TH_ERRORS
    PLAIN(n_args == 7);
    const at::Tensor *const x = gpu_tensor(a[0]), *const codes = gpu_tensor(a[1]), *const w_sc = gpu_tensor(a[2]);
    PLAIN(x && codes && w_sc && dense(*x) && x->dim() > 0 && x->scalar_type() == at::kBFloat16 && codes->device() == x->device() && w_sc->device() == x->device());
    PLAIN(codes->is_contiguous() && w_sc->is_contiguous() && codes->scalar_type() == at::kByte && w_sc->scalar_type() == at::kInt);
    long we, wm, N;
    PLAIN(whole(a[3], we) && whole(a[4], wm) && whole(a[5], N));
    const int64_t K = x->size(-1), M = K > 0 ? x->numel() / K : 0;
    PLAIN(M > 0 && N > 0 && K < (1 << 27));
    const int64_t code_bytes = mase_hip_packed_weight_bytes(N, K, (int)we, (int)wm);
    PLAIN(code_bytes > 0 && codes->numel() == code_bytes && w_sc->numel() == K / 128 * ((N + 255) / 256 * 256));
    LinearRest r;
    PLAIN(linear_rest(*x, N, a[6], r));
    const void* const data = x->data_ptr();
    const uint8_t* const code_data = codes->data_ptr<uint8_t>();
    const uint32_t* const scale_data = reinterpret_cast<const uint32_t*>(w_sc->data_ptr<int>());
    const at::Device device = x->device();
    at::Tensor workspace, y;
    int rc = -1;
    {
        const WithoutGil released;
        const int64_t bytes = mase_hip_mxfp_packed_dense_workspace_bytes(M, N, K);
        if (bytes > 0) workspace = empty({bytes}, at::kByte, device);
        y = empty(r.shape, at::kBFloat16, device);
        rc = mase_hip_mxfp_gemm_packed_dense(data, code_data, scale_data, (int)we, (int)wm, r.bias, r.bias_dtype, y.data_ptr(), M, N, K, bytes > 0 ? workspace.data_ptr() : nullptr, bytes,
                                             r.stream);
    }
    PLAIN(rc == 0);
    return THPVariable_Wrap(std::move(y));
    END_HANDLE_TH_ERRORS
}

// scores(left [.., M, K], right [.., K, N], format of both): left @ right where both are bf16 with the same leading axes and right is the
// transposed view of a contiguous tensor, K up to 128, whichever way is the fastest
PyObject* scores(PyObject*, PyObject* const* a, Py_ssize_t n_args) {
    HANDLE_TH_ERRORS
    PLAIN(n_args == 3);
    const at::Tensor *const l = gpu_tensor(a[0]), *const r = gpu_tensor(a[1]);
    long f[5];
    PLAIN(l && r && ints(a[2], f) && f[0] == 32 && f[3] == 1 && f[4] == 0);
    const int64_t nd = l->dim();
    PLAIN(nd >= 2 && r->dim() == nd && l->scalar_type() == at::kBFloat16 && r->scalar_type() == at::kBFloat16 && l->device() == r->device() && dense(*l) &&
          reinterpret_cast<uintptr_t>(r->data_ptr()) % 16 == 0);
    const int64_t M = l->size(-2), K = l->size(-1), N = r->size(-1);
    PLAIN(r->size(-2) == K && K > 0 && K <= 128 && K % 32 == 0 && N > 0 && N % 8 == 0 && N <= (1 << 23) && M > 0 && l->numel() > 0);
    PLAIN(r->stride(-2) == 1 && (r->stride(-1) == K || N == 1));
    int64_t batches = 1;
    for (int64_t i = nd - 3; i >= 0; --i) {
        PLAIN(l->size(i) == r->size(i) && (l->size(i) == 1 || r->stride(i) == batches * N * K));
        batches *= l->size(i);
    }
    const int way = mase_hip_mxfp_scores_plan(M, N, K, batches, 1), E = (int)f[1], m = (int)f[2];
    void* stream;
    PLAIN((way != 0 || batches <= 65535) && stream_of(*l, &stream));
    Sizes shape = sizes_of(*l);
    shape.back() = N;
    const void *const left = l->data_ptr(), *const right = r->data_ptr();
    const at::Device device = l->device();
    const int64_t n_a = l->numel(), n_w = batches * N * K;
    at::Tensor a_q, w_q, scales, y;
    int rc = 0;
    {
        const WithoutGil released;
        if (way == 0) {
            a_q = empty({n_a}, at::kBFloat16, device);
            scales = empty({n_w / 32}, at::kByte, device);
            w_q = empty({n_w}, at::kByte, device);
            y = empty(shape, at::kBFloat16, device);
            rc = mase_hip_qdq_mxfp(left, 2, a_q.data_ptr(), 2, n_a, 32, E, m, 1, 0, stream);
            if (rc == 0) rc = mase_hip_extract_mxfp(right, 2, scales.data_ptr<uint8_t>(), w_q.data_ptr<uint8_t>(), n_w, 32, E, m, 1, 0, stream);
            if (rc == 0)
                rc = mase_hip_mxfp_gemm_batched(a_q.data_ptr(), 2, scales.data_ptr<uint8_t>(), w_q.data_ptr<uint8_t>(), E, m, y.data_ptr(), 2, M, N, K, 32, batches, M * K, N * K, M * N,
                                                stream);
        } else {
            if (way == 1) {
                w_q = empty({n_w}, at::kBFloat16, device);
                rc = mase_hip_qdq_mxfp(right, 2, w_q.data_ptr(), 2, n_w, 32, E, m, 1, 0, stream);
            }
            if (rc == 0) {
                y = empty(shape, at::kBFloat16, device);
                rc = mase_hip_mxfp_scores(left, E, m, way == 2 ? right : w_q.data_ptr(), way == 2, y.data_ptr(), M, N, K, batches, M * K, N * K, M * N, stream);
            }
        }
    }
    PLAIN(rc == 0);
    return THPVariable_Wrap(std::move(y));
    END_HANDLE_TH_ERRORS
}

// linear_plain(x [.., K], format or None, minifloat, w_scales, w_elements [N * K], exp_bits and frac_bits of W, N, bias or None) -> [.., N] of x's type:
// x quantised to bfloat16 in a pass of its own (None: bfloat16 as it is), then the kernels that compose W's codes
PyObject* linear_plain(PyObject*, PyObject* const* a, Py_ssize_t n_args) {
    HANDLE_TH_ERRORS
    PLAIN(n_args == 9);
    const at::Tensor *const x = gpu_tensor(a[0]), *const w_sc = gpu_tensor(a[3]), *const w_el = gpu_tensor(a[4]);
    PLAIN(x && w_sc && w_el && dense(*x) && x->dim() > 0 && dense(*w_el) && w_sc->is_contiguous() && w_sc->device() == x->device() && w_el->device() == x->device());
    const int dt = dtype_code(x->scalar_type());
    PLAIN((dt == 0 || dt == 2) && w_sc->scalar_type() == at::kByte && w_el->scalar_type() == at::kByte);
    long mini, we, wm, N, f5[5], f4[4];
    PLAIN(whole(a[2], mini) && whole(a[5], we) && whole(a[6], wm) && whole(a[7], N));
    const bool cast = a[1] != Py_None;
    PLAIN(cast ? (mini ? ints(a[1], f4) : ints(a[1], f5)) : dt == 2);
    const int64_t K = x->size(-1), n = x->numel(), M = K > 0 ? n / K : 0;
    PLAIN(M > 0 && N > 0 && N <= INT32_MAX && M <= INT32_MAX && K <= INT32_MAX && K % 32 == 0 && w_el->numel() == N * K && w_sc->numel() == N * K / 32);
    PLAIN(!cast || mini || (f5[0] > 0 && n % f5[0] == 0));
    LinearRest r;
    PLAIN(linear_rest(*x, N, a[8], r));
    const void* const data = x->data_ptr();
    const uint8_t *const scale_data = w_sc->data_ptr<uint8_t>(), *const code_data = w_el->data_ptr<uint8_t>();
    const at::Device device = x->device();
    at::Tensor x_q, workspace, y;
    int rc = 0;
    {
        const WithoutGil released;
        const void* left = data;
        if (cast) {
            x_q = empty({n}, at::kBFloat16, device);
            left = x_q.data_ptr();
            rc = mini ? mase_hip_qdq_minifloat(data, dt, x_q.data_ptr(), 2, n, (int)f4[0], (int)f4[1], (int)f4[2], (int)f4[3], r.stream)
                      : mase_hip_qdq_mxfp(data, dt, x_q.data_ptr(), 2, n, (int)f5[0], (int)f5[1], (int)f5[2], (int)f5[3], (int)f5[4], r.stream);
        }
        if (rc == 0) {
            // (which products are given room for partial sums: kernels._workspace_bytes)
            const bool whole_k = K < (M <= 64 ? 1344 : 1024) && (M <= 64 || N % 128 != 0 || K % 128 != 0);
            const int64_t bytes = whole_k ? 0 : mase_hip_mxfp_gemm_workspace_bytes(1, M, N, K);
            if (bytes > 0) workspace = empty({bytes}, at::kByte, device);
            y = empty(r.shape, kDtypes[dt], device);
            rc = mase_hip_mxfp_gemm_ws(left, 2, nullptr, nullptr, 0, 0, scale_data, code_data, (int)we, (int)wm, r.bias, r.bias_dtype, y.data_ptr(), dt, M, N, K, 32,
                                       bytes > 0 ? workspace.data_ptr() : nullptr, bytes, r.stream);
        }
    }
    PLAIN(rc == 0);
    return THPVariable_Wrap(std::move(y));
    END_HANDLE_TH_ERRORS
}

// Would a product through torch.matmul show `left` more than its values: a graph for its gradient, a tangent, a trace, or autocast's type?
bool followed(const at::Tensor& left) {
    return (at::GradMode::is_enabled() && left.requires_grad()) || left._fw_grad(/*level=*/0).defined() || at::autocast::is_autocast_enabled(at::kCUDA) ||
           torch::jit::tracer::isTracing();
}

// matmul_plain(left [.., M, K], right [.., K, N], format of left or None, format of right): batches of left @ right, the same leading axes on both
// sides, right contiguous or the transposed view of a contiguous tensor: left quantised to bfloat16 (None: bfloat16 as it is), right to
// components in [.., N, K] order, one batched product
PyObject* matmul_plain(PyObject*, PyObject* const* a, Py_ssize_t n_args) {
    HANDLE_TH_ERRORS
    PLAIN(n_args == 4);
    const at::Tensor *const l = gpu_tensor(a[0]), *const r = gpu_tensor(a[1]);
    long fl[5], fr[5];
    PLAIN(l && r && ints(a[3], fr) && fr[0] == 32 && fr[3] == 1);
    const bool cast = a[2] != Py_None;
    const int64_t nd = l->dim();
    const int dt = dtype_code(l->scalar_type());
    PLAIN(nd >= 3 && r->dim() == nd && r->scalar_type() == l->scalar_type() && l->device() == r->device() && dense(*l) && reinterpret_cast<uintptr_t>(r->data_ptr()) % 16 == 0);
    PLAIN(cast ? (dt == 0 || dt == 2) && ints(a[2], fl) && fl[0] > 0 && l->numel() % fl[0] == 0 : dt == 2);
    const int64_t M = l->size(-2), K = l->size(-1), N = r->size(-1);
    PLAIN(r->size(-2) == K && K > 0 && K % 32 == 0 && N > 0 && M > 0 && l->numel() > 0 && M <= INT32_MAX && N <= INT32_MAX && K <= INT32_MAX);
    int64_t batches = 1;
    for (int64_t i = nd - 3; i >= 0; --i) {
        PLAIN(l->size(i) == r->size(i));
        batches *= l->size(i);
    }
    PLAIN(batches > 1 && batches <= 65535);                   // (one matrix: other routes)
    const bool rows = r->is_contiguous();
    if (!rows) {
        PLAIN(!(dt == 2 && K <= 128 && N % 8 == 0));          // (queries and keys: `scores`, or what the wrappers choose for two formats)
        PLAIN(r->stride(-2) == 1 && (r->stride(-1) == K || N == 1));
        int64_t seen = 1;
        for (int64_t i = nd - 3; i >= 0; --i) {
            PLAIN(l->size(i) == 1 || r->stride(i) == seen * N * K);
            seen *= l->size(i);
        }
    }
    // (products whose outputs do not all start on 16 bytes go through torch.matmul otherwise)
    PLAIN((M * N * (dt == 0 ? 4 : 2)) % 16 == 0 || (dt == 2 && N % 16 != 0 && !followed(*l)));
    void* stream;
    PLAIN(stream_of(*l, &stream));
    Sizes shape = sizes_of(*l);
    shape.back() = N;
    const void *const left = l->data_ptr(), *const right = r->data_ptr();
    const at::Device device = l->device();
    const int64_t n_l = l->numel(), n_r = batches * N * K;
    at::Tensor l_q, codes, scales, y;
    int rc = 0;
    {
        const WithoutGil released;
        const void* lq = left;
        // probabilities against values: one format for both, quantised by the product itself
        const bool within = cast && dt == 2 && fl[0] == 32 && fl[1] == fr[1] && fl[2] == fr[2] && fl[3] == 1 && fl[4] == 0 && reinterpret_cast<uintptr_t>(left) % 16 == 0 &&
                            mase_hip_mxfp_matmul_cast_plan(M, N, K);
        if (cast && !within) {
            l_q = empty({n_l}, at::kBFloat16, device);
            lq = l_q.data_ptr();
            rc = mase_hip_qdq_mxfp(left, dt, l_q.data_ptr(), 2, n_l, (int)fl[0], (int)fl[1], (int)fl[2], (int)fl[3], (int)fl[4], stream);
        }
        if (rc == 0) {
            scales = empty({n_r / 32}, at::kByte, device);
            codes = empty({n_r}, at::kByte, device);
            rc = rows ? mase_hip_extract_mxfp_strided(right, dt, scales.data_ptr<uint8_t>(), codes.data_ptr<uint8_t>(), batches, K, N, 32, (int)fr[1], (int)fr[2], 1, (int)fr[4], stream)
                      : mase_hip_extract_mxfp(right, dt, scales.data_ptr<uint8_t>(), codes.data_ptr<uint8_t>(), n_r, 32, (int)fr[1], (int)fr[2], 1, (int)fr[4], stream);
        }
        if (rc == 0) {
            y = empty(shape, kDtypes[dt], device);
            rc = within ? mase_hip_mxfp_matmul_cast(left, scales.data_ptr<uint8_t>(), codes.data_ptr<uint8_t>(), (int)fr[1], (int)fr[2], y.data_ptr(), M, N, K, batches, stream)
                        : mase_hip_mxfp_matmul_batched(lq, scales.data_ptr<uint8_t>(), codes.data_ptr<uint8_t>(), (int)fr[1], (int)fr[2], y.data_ptr(), dt, M, N, K, batches, stream);
        }
    }
    PLAIN(rc == 0);
    return THPVariable_Wrap(std::move(y));
    END_HANDLE_TH_ERRORS
}

#define FN(name) {#name, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)(void)>(name)), METH_FASTCALL, nullptr}
PyMethodDef kMethods[] = {FN(extract_mxfp), FN(qdq_mxfp), FN(compose_mxfp), FN(minifloat), FN(linear_scaled), FN(linear_packed), FN(linear_packed_dense), FN(linear_plain), FN(matmul_plain), FN(scores), {nullptr, nullptr, 0, nullptr}};
PyModuleDef kModule = {PyModuleDef_HEAD_INIT, "_mase_host", nullptr, -1, kMethods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__mase_host(void) {
    PyObject* const c = PyImport_ImportModule("torch._C");
    if (!c) return nullptr;
    g_raw_stream = PyObject_GetAttrString(c, "_cuda_getCurrentRawStream");
    Py_DECREF(c);
    if (!g_raw_stream) return nullptr;
    PyObject* const module = PyModule_Create(&kModule);
    if (module && PyModule_AddStringConstant(module, "built_for", MASE_BUILT_FOR) < 0) {
        Py_DECREF(module);
        return nullptr;
    }
    return module;
}
