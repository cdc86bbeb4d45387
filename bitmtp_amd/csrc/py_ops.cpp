// _bonsai_py: the operators of bitmtp_amd/ops.py from the tensors' handles to the C ABI without
// Python in between.  A decode-width projection runs 3-8 us on the GPU; with checks, allocation,
// device guard and ctypes conversion in Python a call took 11.7 us (37.7 us for a grouped call of
// seven, 46.6 us for the four calls of an MLP block), so back-to-back calls were bound by the host.
// Here a call is one allocation per result plus the launch: 4.2 us for a one-token projection, 9.1 us
// for the seven of a layer, 18.1 us for the MLP block.
//
// Every function returns None when its operands are anything but the plain case (tensor
// subclasses, other devices, dtypes or layouts, shapes the checks refuse, an active dispatch
// mode): the caller then takes its own checked path, which raises the error messages of the
// operator contract.  Nothing is launched before that decision.
#include <Python.h>

#include <ATen/ATen.h>
#include <ATen/hip/EmptyTensor.h>
#include <c10/core/DeviceGuard.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <c10/hip/HIPFunctions.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include <optional>
#include <string>
#include <vector>

#include "../../include/bonsai_decode.h"
#include "../../include/bonsai_gemv.h"

namespace {

constexpr int64_t kMaxOutputs = 1 << 30, kMaxK = 65536;  // the native launchers' limits

// The tensor behind a Python object that is exactly torch.Tensor (or a Parameter), else null.
const at::Tensor *plain(PyObject *o) {
    return THPVariable_CheckExact(o) ? &THPVariable_Unpack(o) : nullptr;
}

bool on_gpu(const at::Tensor &t, c10::Device dev) {
    return t.is_cuda() && t.device() == dev && t.is_contiguous();
}

at::Tensor new_tensor(at::IntArrayRef sizes, at::ScalarType dtype, c10::Device dev) {
    return at::Tensor(at::detail::empty_cuda(sizes, dtype, dev, std::nullopt));
}

// The current device moved to `dev` for the call, where it is another one.
struct OnDevice {
    c10::OptionalDeviceGuard guard;
    explicit OnDevice(c10::Device dev) {
        if (c10::hip::current_device() != dev.index()) guard.reset_device(dev);
    }
    void *stream() const { return c10::hip::getCurrentHIPStream().stream(); }
};

struct ReleaseGil {
    PyThreadState *state = PyEval_SaveThread();
    ~ReleaseGil() { PyEval_RestoreThread(state); }
};

struct Problem {
    int64_t m, n, k;
    bool f16_scales;
};

// The operand checks of a packed projection (bf16 result); false = take the caller's path.
bool gemv_ok(int bits, const at::Tensor &a, const at::Tensor &b, const at::Tensor &s, const at::Tensor &ws,
             bool allow_f16_scales, Problem &p) {
    const int64_t rank = a.dim();
    if ((rank != 2 && rank != 3) || b.dim() != 2 || ws.dim() != 2 || s.dim() < 1) return false;
    const c10::Device dev = a.device();
    if (!on_gpu(a, dev) || !on_gpu(b, dev) || !on_gpu(s, dev) || !on_gpu(ws, dev)) return false;
    if (a.scalar_type() != at::kChar || b.scalar_type() != at::kChar || s.scalar_type() != at::kFloat) return false;
    p.f16_scales = ws.scalar_type() == at::kHalf;
    if (!(ws.scalar_type() == at::kBFloat16 || (allow_f16_scales && p.f16_scales))) return false;
    p.k = a.size(-1);
    p.n = b.size(0);
    if (p.k < 128 || p.k % 128 != 0 || p.k > kMaxK || p.n < 1 || b.size(1) * (8 / bits) != p.k) return false;
    p.m = a.numel() / p.k;
    if (p.m < 1 || p.m * p.n > kMaxOutputs) return false;
    return ws.size(0) == p.n && ws.size(1) == p.k / 128 && s.size(-1) == 1 && s.numel() == p.m;
}

PyObject *fail(const std::string &what) {
    PyErr_SetString(PyExc_RuntimeError, what.c_str());
    return nullptr;
}

const char *kind_name(int bits) { return bits == 2 ? "t2g128" : "q1"; }

// linear(bits, a_int8, b_packed, s, ws, allow_f16_scales) -> bf16 [.., N] or None
PyObject *linear(PyObject *, PyObject *const *args, Py_ssize_t nargs) {
    HANDLE_TH_ERRORS
    if (nargs != 6 || c10::impl::dispatch_mode_enabled()) Py_RETURN_NONE;
    const int bits = (int)PyLong_AsLong(args[0]);
    const at::Tensor *a = plain(args[1]), *b = plain(args[2]), *s = plain(args[3]), *ws = plain(args[4]);
    Problem p;
    if (!a || !b || !s || !ws || !gemv_ok(bits, *a, *b, *s, *ws, args[5] == Py_True, p)) Py_RETURN_NONE;
    if (args[5] == Py_True && a->dim() != 2) Py_RETURN_NONE;
    int64_t shape[3] = {a->size(0), p.n, p.n};
    if (a->dim() == 3) shape[1] = a->size(1);
    at::Tensor out = new_tensor(at::IntArrayRef(shape, a->dim()), at::kBFloat16, a->device());
    const OnDevice on(a->device());
    int rc;
    {
        ReleaseGil unlocked;
        rc = (bits == 2 ? t2g128_gemv_ex : q1g128_gemv_ex)(
            static_cast<const int8_t *>(a->const_data_ptr()), static_cast<const uint8_t *>(b->const_data_ptr()),
            out.mutable_data_ptr(), static_cast<const float *>(s->const_data_ptr()), ws->const_data_ptr(), (int)p.m,
            (int)p.n, (int)p.k, BONSAI_OUT_BF16, p.f16_scales ? BONSAI_SCALE_F16 : BONSAI_SCALE_BF16, on.stream());
    }
    if (rc != 0)
        return fail(std::string(kind_name(bits)) + ": native launch failed with status " + std::to_string(rc) + " (M=" +
                    std::to_string(p.m) + ", N=" + std::to_string(p.n) + ", K=" + std::to_string(p.k) + ")");
    return THPVariable_Wrap(std::move(out));
    END_HANDLE_TH_ERRORS
}

// grouped(bits, problems) -> list of bf16 [M_i, N_i] or None; problems: a list or tuple of 4-tuples
PyObject *grouped(PyObject *, PyObject *const *args, Py_ssize_t nargs) {
    HANDLE_TH_ERRORS
    if (nargs != 2 || c10::impl::dispatch_mode_enabled()) Py_RETURN_NONE;
    const int bits = (int)PyLong_AsLong(args[0]);
    PyObject *seq = args[1];
    if (!PyList_CheckExact(seq) && !PyTuple_CheckExact(seq)) Py_RETURN_NONE;
    const Py_ssize_t count = PySequence_Fast_GET_SIZE(seq);
    if (count < 1 || count > BONSAI_GROUPED_MAX) Py_RETURN_NONE;
    bonsai_gemv_desc descs[BONSAI_GROUPED_MAX];
    const at::Tensor *first = nullptr;
    bool f16 = false;
    for (Py_ssize_t i = 0; i < count; ++i) {
        PyObject *t = PySequence_Fast_GET_ITEM(seq, i);
        if (!PyTuple_CheckExact(t) || PyTuple_GET_SIZE(t) != 4) Py_RETURN_NONE;
        const at::Tensor *a = plain(PyTuple_GET_ITEM(t, 0)), *b = plain(PyTuple_GET_ITEM(t, 1)),
                         *s = plain(PyTuple_GET_ITEM(t, 2)), *ws = plain(PyTuple_GET_ITEM(t, 3));
        Problem p;
        if (!a || !b || !s || !ws || a->dim() != 2 || !gemv_ok(bits, *a, *b, *s, *ws, true, p)) Py_RETURN_NONE;
        if (i == 0) {
            first = a;
            f16 = p.f16_scales;
        } else if (a->device() != first->device() || p.f16_scales != f16) {
            Py_RETURN_NONE;
        }
        descs[i] = {static_cast<const int8_t *>(a->const_data_ptr()), static_cast<const uint8_t *>(b->const_data_ptr()),
                    nullptr, static_cast<const float *>(s->const_data_ptr()), ws->const_data_ptr(), (int32_t)p.m,
                    (int32_t)p.n, (int32_t)p.k, 0};
    }
    PyObject *list = PyList_New(count);
    if (list == nullptr) return nullptr;
    for (Py_ssize_t i = 0; i < count; ++i) {
        const int64_t shape[2] = {descs[i].M, descs[i].N};
        at::Tensor out = new_tensor(at::IntArrayRef(shape, 2), at::kBFloat16, first->device());
        descs[i].out = out.mutable_data_ptr();
        PyList_SET_ITEM(list, i, THPVariable_Wrap(std::move(out)));
    }
    const OnDevice on(first->device());
    int rc;
    {
        ReleaseGil unlocked;
        rc = (bits == 2 ? t2g128_gemv_grouped : q1g128_gemv_grouped)(
            descs, (int)count, BONSAI_OUT_BF16, f16 ? BONSAI_SCALE_F16 : BONSAI_SCALE_BF16, on.stream());
    }
    if (rc != 0) {
        Py_DECREF(list);
        return fail(std::string(kind_name(bits)) + ": grouped native launch failed with status " + std::to_string(rc));
    }
    return list;
    END_HANDLE_TH_ERRORS
}

// q int8 [.., K] and s fp32 [.., 1] of a row-wise quantiser over `x`, K columns kept of each row
struct Quantised {
    at::Tensor q, s;
    Quantised(const at::Tensor &x, int64_t k) {
        c10::SmallVector<int64_t, 4> shape(x.sizes().begin(), x.sizes().end());
        shape.back() = k;
        q = new_tensor(shape, at::kChar, x.device());
        shape.back() = 1;
        s = new_tensor(shape, at::kFloat, x.device());
    }
    int8_t *qp() { return static_cast<int8_t *>(q.mutable_data_ptr()); }
    float *sp() { return static_cast<float *>(s.mutable_data_ptr()); }
};

PyObject *tuple2(at::Tensor a, at::Tensor b) {
    PyObject *t = PyTuple_New(2);
    if (t == nullptr) return nullptr;
    PyTuple_SET_ITEM(t, 0, THPVariable_Wrap(std::move(a)));
    PyTuple_SET_ITEM(t, 1, THPVariable_Wrap(std::move(b)));
    return t;
}

bool rows_ok(const at::Tensor &x, int64_t multiple, int64_t &m, int64_t &k) {
    if (x.dim() < 1 || !x.is_cuda() || !x.is_contiguous()) return false;
    k = x.size(-1);
    if (k < 1 || k % multiple != 0 || k > (1 << 30)) return false;
    m = x.numel() / k;
    return m >= 1 && m <= (1 << 30);
}

// quant_input(x) -> (q, s) or None
PyObject *quant_input(PyObject *, PyObject *x_obj) {
    HANDLE_TH_ERRORS
    const at::Tensor *x = plain(x_obj);
    int64_t m, k;
    if (!x || c10::impl::dispatch_mode_enabled() || !rows_ok(*x, 8, m, k)) Py_RETURN_NONE;
    int kind;
    switch (x->scalar_type()) {
        case at::kBFloat16: kind = BONSAI_X_BF16; break;
        case at::kHalf: kind = BONSAI_X_F16; break;
        case at::kFloat: kind = BONSAI_X_F32; break;
        default: Py_RETURN_NONE;
    }
    Quantised out(*x, k);
    const OnDevice on(x->device());
    int rc;
    {
        ReleaseGil unlocked;
        rc = bonsai_act_quant_int8(x->const_data_ptr(), kind, out.qp(), out.sp(), (int)m, (int)k, on.stream());
    }
    if (rc != 0) return fail("quant_input: native launch failed with status " + std::to_string(rc));
    return tuple2(std::move(out.q), std::move(out.s));
    END_HANDLE_TH_ERRORS
}

bool bf16_on(const at::Tensor &t, c10::Device dev) { return t.scalar_type() == at::kBFloat16 && on_gpu(t, dev); }

// norm_quant(x, w, eps) -> (q, s) or None
PyObject *norm_quant(PyObject *, PyObject *const *args, Py_ssize_t nargs) {
    HANDLE_TH_ERRORS
    if (nargs != 3 || c10::impl::dispatch_mode_enabled() || !PyFloat_CheckExact(args[2])) Py_RETURN_NONE;
    const at::Tensor *x = plain(args[0]), *w = plain(args[1]);
    int64_t m, k;
    if (!x || !w || !rows_ok(*x, 8, m, k) || !bf16_on(*x, x->device()) || !bf16_on(*w, x->device()) || w->dim() != 1 ||
        w->size(0) != k)
        Py_RETURN_NONE;
    Quantised out(*x, k);
    const OnDevice on(x->device());
    int rc;
    {
        ReleaseGil unlocked;
        rc = bonsai_rmsnorm_quant_int8(x->const_data_ptr(), w->const_data_ptr(), (float)PyFloat_AS_DOUBLE(args[2]),
                                       out.qp(), out.sp(), (int)m, (int)k, on.stream());
    }
    if (rc != 0) return fail("fused_norm_quant: native launch failed with status " + std::to_string(rc));
    return tuple2(std::move(out.q), std::move(out.s));
    END_HANDLE_TH_ERRORS
}

// add_norm_quant(x, residual, w, eps) -> (h, q, s) or None
PyObject *add_norm_quant(PyObject *, PyObject *const *args, Py_ssize_t nargs) {
    HANDLE_TH_ERRORS
    if (nargs != 4 || c10::impl::dispatch_mode_enabled() || !PyFloat_CheckExact(args[3])) Py_RETURN_NONE;
    const at::Tensor *x = plain(args[0]), *r = plain(args[1]), *w = plain(args[2]);
    int64_t m, k;
    if (!x || !r || !w || !rows_ok(*x, 8, m, k) || !bf16_on(*x, x->device()) || !bf16_on(*r, x->device()) ||
        !bf16_on(*w, x->device()) || r->sizes() != x->sizes() || w->dim() != 1 || w->size(0) != k)
        Py_RETURN_NONE;
    at::Tensor h = new_tensor(x->sizes(), at::kBFloat16, x->device());
    Quantised out(*x, k);
    const OnDevice on(x->device());
    int rc;
    {
        ReleaseGil unlocked;
        rc = bonsai_add_rmsnorm_quant_int8(x->const_data_ptr(), r->const_data_ptr(), w->const_data_ptr(),
                                           (float)PyFloat_AS_DOUBLE(args[3]), h.mutable_data_ptr(), out.qp(), out.sp(),
                                           (int)m, (int)k, on.stream());
    }
    if (rc != 0) return fail("fused_add_norm_quant: native launch failed with status " + std::to_string(rc));
    PyObject *t = PyTuple_New(3);
    if (t == nullptr) return nullptr;
    PyTuple_SET_ITEM(t, 0, THPVariable_Wrap(std::move(h)));
    PyTuple_SET_ITEM(t, 1, THPVariable_Wrap(std::move(out.q)));
    PyTuple_SET_ITEM(t, 2, THPVariable_Wrap(std::move(out.s)));
    return t;
    END_HANDLE_TH_ERRORS
}

// silu_mul_quant(gate_up) -> (q, s) or None
PyObject *silu_mul_quant(PyObject *, PyObject *x_obj) {
    HANDLE_TH_ERRORS
    const at::Tensor *x = plain(x_obj);
    int64_t m, f2;
    if (!x || c10::impl::dispatch_mode_enabled() || !rows_ok(*x, 16, m, f2) || !bf16_on(*x, x->device())) Py_RETURN_NONE;
    Quantised out(*x, f2 / 2);
    const OnDevice on(x->device());
    int rc;
    {
        ReleaseGil unlocked;
        rc = bonsai_silu_mul_quant_int8(x->const_data_ptr(), out.qp(), out.sp(), (int)m, (int)(f2 / 2), on.stream());
    }
    if (rc != 0) return fail("silu_mul_quant: native launch failed with status " + std::to_string(rc));
    return tuple2(std::move(out.q), std::move(out.s));
    END_HANDLE_TH_ERRORS
}

// prefill_layers(device, dims, eps, scale, buffers, layers) -> 0 / 1: the layers of a decoder over a block
// of prompt rows, ten launches each from one call (a launch costs the stream 2.5-3 us, a ctypes call as
// much again).  Addresses and sizes as Python integers, laid out by bitmtp_amd/model.py:
//   dims     (bits, M, base, dim, n_heads, n_kv, ffn, slots, max_pos, layers, kv_address)
//   buffers  (h0, h1, a_q, a_s, xqkv, q, attn, o_q, o_s, proj, gate_up, i_q, i_s, positions, cos, sin)
//   layers   per layer (wqkv, its scales, wo, scales, gate|up, scales, down, scales, input norm,
//            post-attention norm, q norm, k norm)
// Returns which of h0 / h1 holds the residual stream; the last MLP's output, still to be added, is in proj.
PyObject *prefill_layers(PyObject *, PyObject *const *args, Py_ssize_t nargs) {
    HANDLE_TH_ERRORS
    constexpr int kDims = 11, kBufs = 16, kPerLayer = 12;
    if (nargs != 6 || !PyTuple_CheckExact(args[1]) || PyTuple_GET_SIZE(args[1]) != kDims ||
        !PyTuple_CheckExact(args[4]) || PyTuple_GET_SIZE(args[4]) != kBufs || !PyList_CheckExact(args[5]))
        return fail("prefill_layers: bad arguments");
    long long d[kDims];
    for (int i = 0; i < kDims; ++i) d[i] = PyLong_AsLongLong(PyTuple_GET_ITEM(args[1], i));
    const int bits = (int)d[0], M = (int)d[1], base = (int)d[2], dim = (int)d[3], nh = (int)d[4], nkv = (int)d[5],
              ffn = (int)d[6], slots = (int)d[7], max_pos = (int)d[8], n_layers = (int)d[9];
    const float eps = (float)PyFloat_AsDouble(args[2]), scale = (float)PyFloat_AsDouble(args[3]);
    char *b[kBufs];
    for (int i = 0; i < kBufs; ++i) b[i] = static_cast<char *>(PyLong_AsVoidPtr(PyTuple_GET_ITEM(args[4], i)));
    const Py_ssize_t count = PyList_GET_SIZE(args[5]);
    std::vector<void *> w((size_t)count * kPerLayer);
    for (Py_ssize_t l = 0; l < count; ++l) {
        PyObject *t = PyList_GET_ITEM(args[5], l);
        if (!PyTuple_CheckExact(t) || PyTuple_GET_SIZE(t) != kPerLayer) return fail("prefill_layers: bad layer");
        for (int i = 0; i < kPerLayer; ++i) w[l * kPerLayer + i] = PyLong_AsVoidPtr(PyTuple_GET_ITEM(t, i));
    }
    if (PyErr_Occurred()) return nullptr;
    if (count != n_layers) return fail("prefill_layers: layer count mismatch");
    char *kv = reinterpret_cast<char *>(d[10]);
    const long long head_bytes = (long long)slots * 256, layer_bytes = head_bytes * nkv;
    const int q_dim = nh * BONSAI_HEAD_DIM, qkv = (nh + 2 * nkv) * BONSAI_HEAD_DIM;
    const OnDevice on(c10::Device(c10::DeviceType::CUDA, (c10::DeviceIndex)PyLong_AsLong(args[0])));
    void *st = on.stream();
    int cur = 0;
    const char *what = nullptr;
    int rc = 0;
    {
        ReleaseGil unlocked;
        const auto gemv = bits == 2 ? t2g128_gemv_ex : q1g128_gemv_ex;
        const auto project = [&](char *a, char *s, void *wq, void *ws, char *out, int n, int k) {
            return gemv(reinterpret_cast<const int8_t *>(a), static_cast<const uint8_t *>(wq), out,
                        reinterpret_cast<const float *>(s), ws, M, n, k, BONSAI_OUT_BF16, BONSAI_SCALE_BF16, st);
        };
        char *h[2] = {b[0], b[1]};
        char *a_q = b[2], *a_s = b[3], *xqkv = b[4], *q = b[5], *attn = b[6], *o_q = b[7], *o_s = b[8], *proj = b[9],
             *gu = b[10], *i_q = b[11], *i_s = b[12];
        // T2: activations in operand order where the wide kernel takes them so (what is asked is what is launched later)
        const auto wide = [&](char *a, char *s, void *wq, void *ws, char *out, int n, int k, bool silu, bool ask) {
            return t2g128_gemv_ordered(reinterpret_cast<const int8_t *>(a), static_cast<const uint8_t *>(wq), out,
                                       reinterpret_cast<const float *>(s), ws, M, n, k, silu, ask, st);
        };
        struct {
            bool known, qkv, o, pairs, down;
        } takes = {};
        const auto i8 = [](char *p) { return reinterpret_cast<int8_t *>(p); };
        const auto f32 = [](char *p) { return reinterpret_cast<float *>(p); };
        for (int l = 0; l < n_layers && rc == 0; ++l) {
            void **x = w.data() + (size_t)l * kPerLayer;
            char *kl = kv + l * layer_bytes, *vl = kv + (n_layers + l) * layer_bytes;
#define STEP(name, call)          \
    do {                          \
        if (rc == 0) {            \
            rc = (call);          \
            if (rc != 0) what = name; \
        }                         \
    } while (0)
            // the answers depend on sizes and alignment: those of one aligned layer are those of all (112 asked for in
            // front of 280 launches cost a short prompt, which waits for the host, 1.5 %)
            uintptr_t low = 0;
            for (int i = 0; i < 8; ++i) low |= reinterpret_cast<uintptr_t>(x[i]) & 15;
            if (bits == 2 && (low != 0 || !takes.known)) {
                takes.qkv = wide(a_q, a_s, x[0], x[1], xqkv, qkv, dim, false, true) == 0;
                takes.o = wide(o_q, o_s, x[2], x[3], proj, dim, q_dim, false, true) == 0;
                takes.pairs = wide(a_q, a_s, x[4], x[5], gu, 2 * ffn, dim, true, true) == 0;
                takes.down = takes.pairs && wide(i_q, i_s, x[6], x[7], proj, dim, ffn, false, true) == 0;
                takes.known = low == 0;
            }
            if (takes.qkv) {
                STEP("norm", bonsai_norm_quant_ordered(l == 0 ? h[0] : proj, l == 0 ? nullptr : h[cur], x[8], eps,
                                                       l == 0 ? nullptr : h[cur ^ 1], i8(a_q), f32(a_s), M, dim, st));
                STEP("q|k|v", wide(a_q, a_s, x[0], x[1], xqkv, qkv, dim, false, false));
            } else {
                if (l == 0)
                    STEP("norm", bonsai_rmsnorm_quant_int8(h[0], x[8], eps, i8(a_q), f32(a_s), M, dim, st));
                else
                    STEP("norm", bonsai_add_rmsnorm_quant_int8(proj, h[cur], x[8], eps, h[cur ^ 1], i8(a_q), f32(a_s), M, dim, st));
                STEP("q|k|v", project(a_q, a_s, x[0], x[1], xqkv, qkv, dim));
            }
            if (l != 0) cur ^= 1;
            STEP("rope", bonsai_prefill_rope_kv_write(xqkv, x[10], x[11], eps, b[14], b[15],
                                                      reinterpret_cast<const int32_t *>(b[13]), q, kl, vl, M, nh, nkv,
                                                      slots, base, max_pos, st));
            STEP("attention", bonsai_prefill_attention(q, kl, vl, attn, scale, M, nh, nkv, slots, base, st));
            if (takes.o) {
                STEP("quantiser", bonsai_act_quant_ordered(attn, i8(o_q), f32(o_s), M, q_dim, st));
                STEP("o", wide(o_q, o_s, x[2], x[3], proj, dim, q_dim, false, false));
            } else {
                STEP("quantiser", bonsai_act_quant_int8(attn, BONSAI_X_BF16, i8(o_q), f32(o_s), M, q_dim, st));
                STEP("o", project(o_q, o_s, x[2], x[3], proj, dim, q_dim));
            }
            if (takes.pairs)
                STEP("norm", bonsai_norm_quant_ordered(h[cur], proj, x[9], eps, h[cur ^ 1], i8(a_q), f32(a_s), M, dim, st));
            else
                STEP("norm", bonsai_add_rmsnorm_quant_int8(h[cur], proj, x[9], eps, h[cur ^ 1], i8(a_q), f32(a_s), M, dim, st));
            cur ^= 1;
            // silu(gate) * up leaves with the projection where the wide kernel takes it: half the bytes
            if (takes.pairs) {
                STEP("gate|up", wide(a_q, a_s, x[4], x[5], gu, 2 * ffn, dim, true, false));
                if (takes.down)
                    STEP("quantiser", bonsai_act_quant_ordered(gu, i8(i_q), f32(i_s), M, ffn, st));
                else
                    STEP("quantiser", bonsai_act_quant_int8(gu, BONSAI_X_BF16, i8(i_q), f32(i_s), M, ffn, st));
            } else if (rc == 0) {
                rc = (bits == 2 ? t2g128_gemv_silu : q1g128_gemv_silu)(i8(a_q), static_cast<const uint8_t *>(x[4]), gu, f32(a_s), x[5], M,
                                                                       2 * ffn, dim, st);
                if (rc == 0) {
                    STEP("quantiser", bonsai_act_quant_int8(gu, BONSAI_X_BF16, i8(i_q), f32(i_s), M, ffn, st));
                } else if (rc == -1) {
                    rc = 0;
                    STEP("gate|up", project(a_q, a_s, x[4], x[5], gu, 2 * ffn, dim));
                    STEP("silu", bonsai_silu_mul_quant_int8(gu, i8(i_q), f32(i_s), M, ffn, st));
                } else {
                    what = "gate|up";
                }
            }
            if (takes.down)
                STEP("down", wide(i_q, i_s, x[6], x[7], proj, dim, ffn, false, false));
            else
                STEP("down", project(i_q, i_s, x[6], x[7], proj, dim, ffn));
#undef STEP
        }
    }
    if (rc != 0) return fail(std::string("prompt block: ") + what + " failed with status " + std::to_string(rc));
    return PyLong_FromLong(cur);
    END_HANDLE_TH_ERRORS
}

#define FASTCALL(f) reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)(void)>(f)), METH_FASTCALL
PyMethodDef kMethods[] = {
    {"linear", FASTCALL(linear), "(bits, a_int8, b_packed, s, ws, allow_f16_scales) -> bf16 or None"},
    {"grouped", FASTCALL(grouped), "(bits, [(a_int8, b_packed, s, ws), ...]) -> [bf16, ...] or None"},
    {"quant_input", quant_input, METH_O, "(x) -> (q, s) or None"},
    {"norm_quant", FASTCALL(norm_quant), "(x, w, eps) -> (q, s) or None"},
    {"add_norm_quant", FASTCALL(add_norm_quant), "(x, residual, w, eps) -> (h, q, s) or None"},
    {"prefill_layers", FASTCALL(prefill_layers), "(device, dims, eps, scale, buffers, layers) -> residual buffer"},
    {"silu_mul_quant", silu_mul_quant, METH_O, "(gate_up) -> (q, s) or None"},
    {nullptr, nullptr, 0, nullptr}};
PyModuleDef kModule = {PyModuleDef_HEAD_INIT, "_bonsai_py", nullptr, -1, kMethods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__bonsai_py(void) { return PyModule_Create(&kModule); }
