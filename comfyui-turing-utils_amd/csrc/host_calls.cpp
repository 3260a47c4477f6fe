// The whole host side of the three hot calls as one native function each:
// checks, output and scratch tensors, launches.
//
// A short call is bound by its host work, not by its kernels: from Python the
// W8A8 linear of one row spent 42 us on the host (two dispatched custom ops,
// three tensors and eight argument normalisations in the interpreter) for 10 us
// of kernels, Sage attention over 257 tokens 51 us for 20.  Here the same work
// takes 6-10 us and hides behind the kernels of the call before.
//
// Each function serves the plain form of its call only: dense contiguous CUDA
// tensors of exactly the kernels' types on the current device, no dispatch or
// function mode, no tracing or functorch transform, nothing that autograd
// would record.  For everything else it returns None, and the caller runs its
// general Python route, which converts, pads, dispatches or raises.  The
// launches are those of the general route, so results have the same bits.
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include <ATen/ATen.h>
#include <ATen/PythonTorchFunctionTLS.h>
#include <c10/core/GradMode.h>
#include <c10/core/impl/DeviceGuardImplInterface.h>
#include <c10/core/impl/LocalDispatchKeySet.h>

#include <cmath>
#include <cstdint>
#include <string>

#include "../../include/tu_hip.h"

namespace {

using at::Tensor;

// A tensor argument is plain when nothing but the CUDA kernel (and autograd,
// which must have nothing to record) would see it.
bool plain(PyObject *obj, const Tensor **out, c10::Device device) {
    if (!THPVariable_CheckTypeExact(Py_TYPE(obj))) return false;
    const Tensor &t = THPVariable_Unpack(obj);
    constexpr c10::DispatchKeySet cuda(c10::DispatchKey::CUDA);
    constexpr c10::DispatchKeySet autograd =
        cuda | c10::DispatchKeySet(c10::DispatchKey::ADInplaceOrView) | c10::DispatchKeySet(c10::DispatchKey::AutogradCUDA);
    // autocast has no rule for any of these calls
    const c10::DispatchKeySet keys = t.key_set() - c10::DispatchKeySet(c10::DispatchKey::AutocastCUDA);
    if (keys != autograd && keys != cuda) return false;
    if (t.device() != device || t.layout() != at::kStrided) return false;
    if (keys == autograd && ((t.requires_grad() && c10::GradMode::is_enabled()) || t._fw_grad(0).defined()))
        return false;
    *out = &t;
    return true;
}

// No mode, transform or tracer is listening, `index` is the current device
// and a supported one.
bool plain_context(int64_t index) {
    constexpr c10::DispatchKeySet usual =
        c10::DispatchKeySet(c10::DispatchKey::BackendSelect) | c10::DispatchKeySet(c10::DispatchKey::ADInplaceOrView);
    const auto included = c10::impl::tls_local_dispatch_key_set().included_;
    if (!(included - usual).empty() || at::impl::torch_function_mode_enabled()) return false;
    const c10::impl::DeviceGuardImplInterface *guard = c10::impl::getDeviceGuardImpl(c10::kCUDA);
    return guard->getDevice().index() == index && tu_device_supported(static_cast<int32_t>(index)) == 1;
}

bool aligned(const Tensor &t, uintptr_t bytes) { return (reinterpret_cast<uintptr_t>(t.data_ptr()) & (bytes - 1)) == 0; }

Tensor empty(at::IntArrayRef sizes, at::ScalarType type, c10::Device device) {
    return at::empty(sizes, at::TensorOptions().dtype(type).device(device));
}

void *ptr(const Tensor &t) { return t.defined() ? t.data_ptr() : nullptr; }

[[noreturn]] void failed(const char *name) {
    throw std::runtime_error(std::string(name) + ": " + tu_last_error());
}

int64_t ceil_div(int64_t a, int64_t b) { return (a + b - 1) / b; }

// An integer argument (bools among them).
bool integer(PyObject *obj, int64_t *out) {
    if (!PyLong_Check(obj)) return false;
    *out = PyLong_AsLongLong(obj);
    if (*out == -1 && PyErr_Occurred()) {
        PyErr_Clear();
        return false;
    }
    return true;
}

struct ReleaseGil {
    PyThreadState *state = PyEval_SaveThread();
    ~ReleaseGil() { PyEval_RestoreThread(state); }
};

// The quantizer's widest row; the general route refuses a wider one with a ValueError.
constexpr int64_t kMaxColumns = 65536;

// int8_linear(x, weight, weight_scale, bias, out_kind, group, act, stream):
// ConvRot quantizer and INT8 GEMM.  out_kind 0 bf16, 1 fp16, 2 fp32.
PyObject *int8_linear(PyObject *, PyObject *const *args, Py_ssize_t nargs) {
    HANDLE_TH_ERRORS
    int64_t kind, group, act, stream;
    if (nargs != 8 || !integer(args[4], &kind) || !integer(args[5], &group) || !integer(args[6], &act) ||
        !integer(args[7], &stream) || !THPVariable_CheckTypeExact(Py_TYPE(args[0])))
        Py_RETURN_NONE;
    const c10::Device device = THPVariable_Unpack(args[0]).device();
    const Tensor *x, *w, *ws, *bias = nullptr;
    if (!device.is_cuda() || !plain_context(device.index()) || !plain(args[0], &x, device) ||
        !plain(args[1], &w, device) || !plain(args[2], &ws, device) ||
        (args[3] != Py_None && !plain(args[3], &bias, device)))
        Py_RETURN_NONE;
    if (x->scalar_type() != at::kBFloat16 || x->dim() < 1 || !x->is_contiguous() || !aligned(*x, 16) ||
        w->scalar_type() != at::kChar || w->dim() != 2 || !w->is_contiguous() || ws->scalar_type() != at::kFloat ||
        !ws->is_contiguous() || (group != 128 && group != 256) || act < 0 || act > 2 || kind < 0 || kind > 2)
        Py_RETURN_NONE;
    const int64_t n = w->size(0), k = w->size(1), width = act == TU_ACT_SWIGLU ? 2 * k : k;
    if (n <= 0 || n % 8 || k <= 0 || k > kMaxColumns || k % group || x->size(-1) != width || x->numel() == 0 || ws->numel() != n ||
        (bias && (bias->scalar_type() != at::kFloat || !bias->is_contiguous() || bias->numel() != n)))
        Py_RETURN_NONE;
    const int64_t m = x->numel() / width;
    Tensor out;
    {
        ReleaseGil nogil;
        c10::SmallVector<int64_t, 4> shape(x->sizes().begin(), x->sizes().end());
        shape.back() = n;
        const Tensor q = empty({m, k}, at::kChar, device), s = empty({m}, at::kFloat, device);
        out = empty(shape, kind == 0 ? at::kBFloat16 : kind == 1 ? at::kHalf : at::kFloat, device);
        void *st = reinterpret_cast<void *>(stream);
        if (tu_convrot_quant_i8(x->data_ptr(), q.data_ptr<int8_t>(), s.data_ptr<float>(), m, k,
                                static_cast<int32_t>(group), static_cast<int32_t>(act), st))
            failed("tu_convrot_quant_i8");
        const int8_t *qp = q.data_ptr<int8_t>(), *wp = w->data_ptr<int8_t>();
        const float *sp = s.data_ptr<float>(), *wsp = ws->data_ptr<float>();
        const float *bp = bias ? bias->data_ptr<float>() : nullptr;
        void *o = out.data_ptr();
        if (kind == 0 && tu_int8_gemm_bf16(qp, wp, sp, wsp, bp, o, m, n, k, st)) failed("tu_int8_gemm_bf16");
        if (kind == 1 && tu_int8_gemm_f16(qp, wp, sp, wsp, bp, o, m, n, k, st)) failed("tu_int8_gemm_f16");
        if (kind == 2 && tu_int8_gemm_f32(qp, wp, sp, wsp, bp, static_cast<float *>(o), m, n, k, st))
            failed("tu_int8_gemm_f32");
    }
    return THPVariable_Wrap(std::move(out));
    END_HANDLE_TH_ERRORS
}

// Sizes and strides of Q / K / V in either layout.
struct Qkv {
    const Tensor *q, *k, *v;
    int64_t batch, hq, hkv, lq, lk, dim;
    int head, seq;  // axes
    int64_t sb(const Tensor &t) const { return t.stride(0); }
    int64_t sh(const Tensor &t) const { return t.stride(head); }
    int64_t sl(const Tensor &t) const { return t.stride(seq); }
};

bool rows_aligned(const Tensor &t) {
    return t.stride(3) == 1 && t.stride(0) % 8 == 0 && t.stride(1) % 8 == 0 && t.stride(2) % 8 == 0 && aligned(t, 16);
}

bool unpack_qkv(PyObject *const *args, bool nhd, Qkv &a) {
    if (!THPVariable_CheckTypeExact(Py_TYPE(args[0]))) return false;
    const c10::Device device = THPVariable_Unpack(args[0]).device();
    if (!device.is_cuda() || !plain_context(device.index()) || !plain(args[0], &a.q, device) ||
        !plain(args[1], &a.k, device) || !plain(args[2], &a.v, device))
        return false;
    const Tensor &q = *a.q, &k = *a.k, &v = *a.v;
    if (q.scalar_type() != k.scalar_type() || q.scalar_type() != v.scalar_type() || q.dim() != 4 || k.dim() != 4 ||
        v.dim() != 4 || k.sizes() != v.sizes())
        return false;
    a.head = nhd ? 2 : 1;
    a.seq = nhd ? 1 : 2;
    a.batch = q.size(0);
    a.hq = q.size(a.head);
    a.lq = q.size(a.seq);
    a.hkv = k.size(a.head);
    a.lk = k.size(a.seq);
    a.dim = q.size(3);
    return (a.dim == 64 || a.dim == 128) && k.size(0) == a.batch && k.size(3) == a.dim && a.batch > 0 && a.hq > 0 &&
           a.lq > 0 && a.lk > 0 && a.hkv > 0 && a.hq % a.hkv == 0 && rows_aligned(q) && rows_aligned(k) &&
           rows_aligned(v);
}

// sageattn(q, k, v, nhd, causal, scale, smooth_k, blkq, blkk, cus, stream)
PyObject *sageattn(PyObject *, PyObject *const *args, Py_ssize_t nargs) {
    HANDLE_TH_ERRORS
    int64_t nhd, causal, smooth, blkq, blkk, cus, stream;
    if (nargs != 11 || !integer(args[3], &nhd) || !integer(args[4], &causal) || !PyFloat_Check(args[5]) ||
        !integer(args[6], &smooth) || !integer(args[7], &blkq) || !integer(args[8], &blkk) || !integer(args[9], &cus) ||
        !integer(args[10], &stream))
        Py_RETURN_NONE;
    const float scale = static_cast<float>(PyFloat_AS_DOUBLE(args[5]));
    Qkv a;
    if (!(scale > 0.0f && std::isfinite(scale)) || (blkq != 16 && blkq != 32 && blkq != 64 && blkq != 128) ||
        (blkk != 64 && blkk != 128) || !unpack_qkv(args, nhd != 0, a) || a.q->scalar_type() != at::kBFloat16)
        Py_RETURN_NONE;
    const int64_t lpad = ceil_div(a.lk, 64) * 64;
    // past the one grid of the shared prologue launch
    if (a.batch * (a.hkv * (lpad / 32) + a.hq * ceil_div(a.lq, blkq)) > 1 << 23) Py_RETURN_NONE;
    Tensor out;
    {
        ReleaseGil nogil;
        const c10::Device device = a.q->device();
        const Tensor q8 = empty(a.q->sizes(), at::kChar, device), k8 = empty(a.k->sizes(), at::kChar, device);
        const Tensor qs = empty({a.batch, a.hq, ceil_div(a.lq, blkq)}, at::kFloat, device);
        const Tensor ks = empty({a.batch, a.hkv, ceil_div(a.lk, blkk)}, at::kFloat, device);
        const Tensor vt = empty({a.batch, a.hkv, a.dim, lpad}, at::kBFloat16, device);
        const int32_t c = causal != 0;
        void *st = reinterpret_cast<void *>(stream);
        {
            const int64_t bytes = tu_sage_prep_workspace(a.batch, a.hkv, a.lk, a.dim, smooth != 0);
            Tensor work;
            if (bytes > 0) work = empty({bytes}, at::kByte, device);
            if (tu_sage_prep(a.q->data_ptr(), a.k->data_ptr(), a.v->data_ptr(), a.batch, a.hq, a.hkv, a.lq, a.lk, a.dim,
                             a.sb(*a.q), a.sh(*a.q), a.sl(*a.q), a.sb(*a.k), a.sh(*a.k), a.sl(*a.k), a.sb(*a.v),
                             a.sh(*a.v), a.sl(*a.v), smooth != 0, blkq, blkk, q8.data_ptr<int8_t>(), a.sb(q8), a.sh(q8),
                             a.sl(q8), k8.data_ptr<int8_t>(), a.sb(k8), a.sh(k8), a.sl(k8), qs.data_ptr<float>(),
                             ks.data_ptr<float>(), vt.data_ptr(), lpad, ptr(work), bytes, st))
                failed("tu_sage_prep");
        }
        out = empty(a.q->sizes(), at::kBFloat16, device);
        const int64_t bytes =
            tu_sage_attn_workspace(a.batch, a.hq, a.lq, a.lk, a.dim, c, static_cast<int32_t>(cus));
        Tensor part;
        if (bytes > 0) part = empty({bytes}, at::kByte, device);
        if (tu_sage_attn_fwd_auto(q8.data_ptr<int8_t>(), qs.data_ptr<float>(), blkq, k8.data_ptr<int8_t>(),
                                  ks.data_ptr<float>(), blkk, vt.data_ptr(), lpad, out.data_ptr(), a.batch, a.hq, a.hkv,
                                  a.lq, a.lk, a.dim, a.sb(q8), a.sh(q8), a.sl(q8), a.sb(k8), a.sh(k8), a.sl(k8),
                                  a.sb(out), a.sh(out), a.sl(out), scale, c, static_cast<int32_t>(cus), ptr(part), bytes,
                                  st))
            failed("tu_sage_attn_fwd_auto");
    }
    return THPVariable_Wrap(std::move(out));
    END_HANDLE_TH_ERRORS
}

// w8a8attn(q, k, v, causal, scale, rotate, stabilize, stream), HND
PyObject *w8a8attn(PyObject *, PyObject *const *args, Py_ssize_t nargs) {
    HANDLE_TH_ERRORS
    int64_t causal, rotate, stabilize, stream;
    if (nargs != 8 || !integer(args[3], &causal) || !PyFloat_Check(args[4]) || !integer(args[5], &rotate) ||
        !integer(args[6], &stabilize) || !integer(args[7], &stream))
        Py_RETURN_NONE;
    const float scale = static_cast<float>(PyFloat_AS_DOUBLE(args[4]));
    Qkv a;
    if (!unpack_qkv(args, false, a)) Py_RETURN_NONE;
    const at::ScalarType type = a.q->scalar_type();
    if (type != at::kBFloat16 && type != at::kHalf) Py_RETURN_NONE;
    Tensor out;
    {
        ReleaseGil nogil;
        const c10::Device device = a.q->device();
        const int64_t lpad = ceil_div(a.lk, 64) * 64, nqs = ceil_div(a.lq, 64) * 4, nks = ceil_div(a.lk, 64);
        const Tensor q8 = empty({a.batch, a.hq, a.lq, 128}, at::kChar, device);
        const Tensor k8 = empty({a.batch, a.hkv, a.lk, 128}, at::kChar, device);
        const Tensor v8 = empty({a.batch, a.hkv, 128, lpad}, at::kChar, device);
        const Tensor qs = empty({a.batch, a.hq, nqs}, at::kFloat, device);
        const Tensor ks = empty({a.batch, a.hkv, nks}, at::kFloat, device);
        const Tensor vs = empty({a.batch, a.hkv, 128}, at::kFloat, device);
        const int32_t f16 = type == at::kHalf;
        void *st = reinterpret_cast<void *>(stream);
        {
            Tensor anchors;
            if (rotate && stabilize) anchors = empty({a.batch, a.hkv}, at::kInt, device);
            const int64_t bytes = tu_w8a8_quant_v_workspace(a.batch, a.hkv, a.lk, a.dim);
            const Tensor work = empty({bytes}, at::kByte, device);
            if (tu_w8a8_prep(a.q->data_ptr(), a.k->data_ptr(), a.v->data_ptr(), f16, a.batch, a.hq, a.hkv, a.lq, a.lk,
                             a.dim, a.sb(*a.q), a.sh(*a.q), a.sl(*a.q), a.sb(*a.k), a.sh(*a.k), a.sl(*a.k), a.sb(*a.v),
                             a.sh(*a.v), a.sl(*a.v), q8.data_ptr<int8_t>(), a.sb(q8), a.sh(q8), a.sl(q8),
                             k8.data_ptr<int8_t>(), a.sb(k8), a.sh(k8), a.sl(k8), qs.data_ptr<float>(),
                             ks.data_ptr<float>(), anchors.defined() ? anchors.data_ptr<int32_t>() : nullptr,
                             rotate != 0, v8.data_ptr<int8_t>(), lpad, vs.data_ptr<float>(), a.dim == 64,
                             work.data_ptr(), bytes, st))
                failed("tu_w8a8_prep");
        }
        out = empty({a.batch, a.hq, a.lq, 128}, type, device);
        if (tu_w8a8_attn_fwd(q8.data_ptr<int8_t>(), qs.data_ptr<float>(), nqs, k8.data_ptr<int8_t>(),
                             ks.data_ptr<float>(), nks, v8.data_ptr<int8_t>(), vs.data_ptr<float>(), lpad,
                             out.data_ptr(), f16, a.batch, a.hq, a.hkv, a.lq, a.lk, 128, a.sb(q8), a.sh(q8), a.sl(q8),
                             a.sb(k8), a.sh(k8), a.sl(k8), a.sb(out), a.sh(out), a.sl(out), scale, causal != 0, st))
            failed("tu_w8a8_attn_fwd");
        if (a.dim == 64) out = out.narrow(3, 0, 64);
    }
    return THPVariable_Wrap(std::move(out));
    END_HANDLE_TH_ERRORS
}

#define TU_METHOD(NAME) \
    {#NAME, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(NAME)), METH_FASTCALL, nullptr}
PyMethodDef methods[] = {TU_METHOD(int8_linear), TU_METHOD(sageattn), TU_METHOD(w8a8attn), {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_host_calls", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

// torch_version: the torch whose headers and libraries this was built against;
// the loader compares it with the running one.
PyMODINIT_FUNC PyInit__host_calls() {
    PyObject *m = PyModule_Create(&module);
    if (m && PyModule_AddStringConstant(m, "torch_version", TU_TORCH_VERSION)) {
        Py_DECREF(m);
        return nullptr;
    }
    return m;
}
