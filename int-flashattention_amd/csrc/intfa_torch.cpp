// The Python entry points' host side: argument checks of the reference wrappers, layout normalisation, output allocation,
// the parameter blocks of include/intfa.h and the launch, as a CPython extension module (`_native`) over libtorch.
//
// What bounds it: a decoding step launches kernels of 2 - 10 us each, so the host has to get from the Python call to the
// launch in about the same time.  The same steps written in Python over ctypes (attribute accesses on tensors, one setattr
// per field, a device context manager, record_stream through the dispatcher) took 28 - 32 us per attention call and 15 - 18 us
// per quantiser call; here the tensors are read through their C++ objects and the arguments arrive by
// vectorcall, without a binding layer in between.
//
// Functions take positional arguments only (the keyword interface and its defaults live in the Python modules).
#include <torch/csrc/Dtype.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include <ATen/Functions.h>
#include <ATen/hip/EmptyTensor.h>
#include <ATen/hip/impl/HIPCachingAllocatorMasqueradingAsCUDA.h>
#include <ATen/hip/impl/HIPGuardImplMasqueradingAsCUDA.h>
#include <ATen/hip/impl/HIPStreamMasqueradingAsCUDA.h>

#include <atomic>
#include <climits>
#include <string>

#include "../../include/intfa.h"

namespace {

using at::ScalarType;
using at::Tensor;

constexpr int kMinHeadDim = 64;     // smaller head dims are zero-padded up to this (QK^T and the kept output columns are unchanged)
constexpr int kBlockM = 128;        // query block of the general kernels
constexpr int kDecodeRows = 64;     // most query rows the decode-shaped kernels take

[[noreturn]] void fail(PyObject* type, const std::string& text) {
    PyErr_SetString(type, text.c_str());
    throw python_error();
}
// A call of the C ABI with the interpreter lock released (a launch blocks while the stream's queue is full).
template <typename F> int unlocked(F call) {
    PyThreadState* const state = PyEval_SaveThread();
    const int rc = call();
    PyEval_RestoreThread(state);
    return rc;
}
void check_rc(int rc, const char* what) {
    if (rc != INTFA_OK)
        fail(PyExc_RuntimeError, std::string(what) + " failed with code " + std::to_string(rc) + ": " + intfa_error_string(rc));
}

// ---- argument conversion
const Tensor& tensor_arg(PyObject* o, const char* name) {
    if (!THPVariable_Check(o)) fail(PyExc_TypeError, std::string(name) + " must be a tensor, got " + Py_TYPE(o)->tp_name);
    return THPVariable_Unpack(o);
}
// None -> an undefined tensor
const Tensor& optional_tensor_arg(PyObject* o, const char* name) {
    static const Tensor none;
    return o == Py_None ? none : tensor_arg(o, name);
}
int64_t int_arg(PyObject* o) {
    const long long v = PyLong_Check(o) ? PyLong_AsLongLong(o) : [&] {
        PyObject* i = PyNumber_Long(o);
        if (i == nullptr) throw python_error();
        const long long r = PyLong_AsLongLong(i);
        Py_DECREF(i);
        return r;
    }();
    if (v == -1 && PyErr_Occurred()) throw python_error();
    return v;
}
int int32_arg(PyObject* o, const char* name) {
    const int64_t v = int_arg(o);
    if (v < INT_MIN || v > INT_MAX) fail(PyExc_ValueError, std::string(name) + " is out of range");
    return (int)v;
}
double float_arg(PyObject* o) {
    const double v = PyFloat_AsDouble(o);
    if (v == -1.0 && PyErr_Occurred()) throw python_error();
    return v;
}
bool bool_arg(PyObject* o) {
    const int v = PyObject_IsTrue(o);
    if (v < 0) throw python_error();
    return v != 0;
}
void expect_args(Py_ssize_t n, Py_ssize_t want, const char* name) {
    if (n != want) fail(PyExc_TypeError, std::string(name) + " takes " + std::to_string(want) + " arguments, got " + std::to_string(n));
}

// ---- tensor helpers
int dtype_enum(ScalarType t) {
    switch (t) {
        case ScalarType::Half: return INTFA_F16;
        case ScalarType::BFloat16: return INTFA_BF16;
        case ScalarType::Float: return INTFA_F32;
        default: return -1;
    }
}
std::string dtype_text(ScalarType t) { return std::string("torch.") + at::toString(t); }

void require_4d(const Tensor& t, const char* name) {
    if (t.dim() != 4) fail(PyExc_ValueError, std::string(name) + " must be a [Z, H, N, d] tensor");
}
void require_gpu(const Tensor& t) {
    if (t.defined() && !t.is_cuda()) fail(PyExc_RuntimeError, "int_flashattention_amd kernels run on the GPU only; got a CPU tensor");
}
// The reference's shape constraints (flash_atten_full_int8.py:189-193).
int64_t head_dim_of(const Tensor& q, const Tensor& k, const Tensor& v) {
    const int64_t hq = q.size(-1), hk = k.size(-1), hv = v.size(-1);
    if (hq != hk || hk != hv) fail(PyExc_AssertionError, "q, k and v must have the same head_dim");
    if (hk != 16 && hk != 32 && hk != 64 && hk != 128 && hk != 256) fail(PyExc_AssertionError, "head_dim must be 16, 32, 64, 128 or 256");
    return hk;
}
// t itself if its head dim is contiguous and every other stride is 16-byte aligned, else a contiguous copy; head dims
// below `d_to` are zero-padded.
Tensor row_major(const Tensor& t, int64_t d_to, int elem_bytes) {
    const Tensor x = t.size(-1) == d_to ? t : at::constant_pad_nd(t, {0, d_to - t.size(-1)});
    bool ok = x.stride(-1) == 1 && reinterpret_cast<uintptr_t>(x.data_ptr()) % 16 == 0;
    for (int64_t i = 0; i + 1 < x.dim(); ++i) ok = ok && (x.stride(i) * elem_bytes) % 16 == 0;
    return ok ? x : x.contiguous();
}
// True if the rows of consecutive heads of t ([Z, H, N, ...]) lie at one constant stride.
bool can_fold(const Tensor& t, int64_t n) { return n == 1 || t.stride(1) == n * t.stride(2); }

// The device of a call made current for its duration, and its current stream.  (The caller's stream: an input that was
// allocated on another one is marked as in use here, so that its memory is not handed out again before this call is done.)
struct CallDevice {
    c10::hip::OptionalHIPGuardMasqueradingAsCUDA guard;
    c10::hip::HIPStreamMasqueradingAsCUDA stream;
    at::Device device;
    explicit CallDevice(const Tensor& t) : guard(t.device()), stream(c10::hip::getCurrentHIPStreamMasqueradingAsCUDA(t.device().index())), device(t.device()) {}
    Tensor empty(at::IntArrayRef size, ScalarType dtype) const { return at::detail::empty_cuda(size, dtype, device, std::nullopt); }
    void* raw_stream() const { return (void*)stream.stream(); }
    void used(const Tensor& t) const {
        if (t.defined()) c10::hip::HIPCachingAllocatorMasqueradingAsCUDA::recordStreamMasqueradingAsCUDA(t.storage().data_ptr(), stream);
    }
};

// compute units of a device, looked up once
int compute_units(int dev) {
    static std::atomic<int> known[64];
    if (dev >= 0 && dev < 64) {
        const int n = known[dev].load(std::memory_order_relaxed);
        if (n > 0) return n;
    }
    int n = 0;
    if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess) n = 0;
    if (dev >= 0 && dev < 64) known[dev].store(n, std::memory_order_relaxed);
    return n;
}

void set_strides(int64_t* dst, const Tensor& t) {      // batch, head, row (three consecutive members of a parameter block)
    dst[0] = t.stride(0); dst[1] = t.stride(1); dst[2] = t.stride(2);
}

// ---- forward(variant, q, k, v, q_scale, k_scale, v_scale, causal, sm_scale, out_dtype, num_splits, p_round, return_lse,
//              v_scale_block, seqlens_k); variant is INTFA_VARIANT_*, num_splits a count or "auto"
PyObject* forward(PyObject*, PyObject* const* a, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    expect_args(n, 15, "forward");
    const int variant = int32_arg(a[0], "variant");
    const bool full = variant == INTFA_VARIANT_FULL_INT8, scaled = variant != INTFA_VARIANT_FP16;
    const Tensor &q = tensor_arg(a[1], "q"), &k = tensor_arg(a[2], "k"), &v = tensor_arg(a[3], "v");
    const Tensor& q_scale = scaled ? tensor_arg(a[4], "q_scale") : optional_tensor_arg(Py_None, "");
    const Tensor& k_scale_in = scaled ? tensor_arg(a[5], "k_scale") : optional_tensor_arg(Py_None, "");
    const Tensor& v_scale_in = full ? tensor_arg(a[6], "v_scale") : optional_tensor_arg(Py_None, "");
    const bool causal = bool_arg(a[7]);
    const float sm_scale = (float)float_arg(a[8]);
    if (!THPDtype_Check(a[9])) fail(PyExc_TypeError, "out_dtype must be a torch.dtype");
    const ScalarType out_type = reinterpret_cast<THPDtype*>(a[9])->scalar_type;
    const int p_round = int32_arg(a[11], "p_round");
    const bool return_lse = bool_arg(a[12]);
    const Tensor& seqlens = optional_tensor_arg(a[14], "seqlens_k");
    for (const Tensor* t : {&q, &k, &v, &q_scale, &k_scale_in, &v_scale_in}) require_gpu(*t);
    require_4d(q, "q"); require_4d(k, "k"); require_4d(v, "v");
    const int64_t d = head_dim_of(q, k, v), dk = d < kMinHeadDim ? kMinHeadDim : d;
    const int64_t Z = q.size(0), H = q.size(1), N = q.size(2), Hkv = k.size(1), Nk = k.size(2);
    if (k.size(0) != Z || v.size(0) != Z || v.size(2) != Nk || v.size(1) != Hkv)
        fail(PyExc_ValueError, "q, k and v must share the batch size, and k and v their heads and length");
    if (Hkv == 0 || H % Hkv != 0)
        fail(PyExc_ValueError, "the number of query heads (" + std::to_string(H) + ") must be a multiple of the number of K/V heads (" + std::to_string(Hkv) + ")");
    const int io_dtype = dtype_enum(out_type);
    if (io_dtype < 0) fail(PyExc_KeyError, dtype_text(out_type));

    const CallDevice dev(q);
    const Tensor q_ = row_major(q, dk, scaled ? 1 : 2), k_ = row_major(k, dk, scaled ? 1 : 2), v_ = row_major(v, dk, full ? 1 : 2);
    Tensor out = dev.empty({Z, H, N, dk}, out_type), lse;
    if (return_lse) lse = dev.empty({Z, H, N}, ScalarType::Float);

    intfa_fwd_params p{};
    p.q = q_.data_ptr(); p.k = k_.data_ptr(); p.v = v_.data_ptr(); p.out = out.data_ptr();
    p.lse = return_lse ? lse.data_ptr<float>() : nullptr;
    set_strides(&p.q_stride_b, q_); set_strides(&p.k_stride_b, k_); set_strides(&p.v_stride_b, v_); set_strides(&p.o_stride_b, out);
    Tensor k_scale, v_scale, seqlens_;
    if (scaled) {
        if (q_scale.dim() != 3 || k_scale_in.dim() != 3) fail(PyExc_ValueError, "q_scale and k_scale must be [Z, H, N] tensors");
        k_scale = k_scale_in.scalar_type() == q_scale.scalar_type() ? k_scale_in : k_scale_in.to(q_scale.scalar_type());
        p.scale_dtype = dtype_enum(q_scale.scalar_type());
        if (p.scale_dtype < 0) fail(PyExc_TypeError, "unsupported scale dtype " + dtype_text(q_scale.scalar_type()));
        p.q_scale = q_scale.data_ptr(); p.k_scale = k_scale.data_ptr();
        set_strides(&p.qs_stride_b, q_scale); set_strides(&p.ks_stride_b, k_scale);
    }
    if (full) {
        if (v_scale_in.dim() == 4) {
            // one scale per block of keys and channel ([Z, H_kv, ceil(N_k / v_scale_block), d]); blocked scales cross the ABI as fp32
            const int64_t vsb = a[13] == Py_None ? intfa_fwd_block_n(variant, (int)dk) : int32_arg(a[13], "v_scale_block");
            v_scale = v_scale_in.to(ScalarType::Float);
            if (vsb <= 0 || v_scale.size(0) != Z || v_scale.size(1) != Hkv || v_scale.size(2) != (Nk + vsb - 1) / vsb || v_scale.size(3) != d)
                fail(PyExc_ValueError, "a blocked v_scale must be [Z, H_kv, ceil(N_k / " + std::to_string(vsb) + "), d], got " +
                                           c10::str(v_scale.sizes()));
            if (d != dk) v_scale = at::constant_pad_nd(v_scale, {0, dk - d});
            if (v_scale.stride(-1) != 1) v_scale = v_scale.contiguous();
            p.v_scale_block = (int)vsb;
            p.vs_stride_b = v_scale.stride(0); p.vs_stride_h = v_scale.stride(1); p.vs_stride_blk = v_scale.stride(2);
        } else {
            if (a[13] != Py_None) fail(PyExc_ValueError, "v_scale_block needs a 4-D v_scale");
            if (v_scale_in.dim() != 2) fail(PyExc_ValueError, "v_scale must be a [Z, H] tensor (or 4-D: one scale per block of keys and channel)");
            v_scale = v_scale_in.scalar_type() == q_scale.scalar_type() ? v_scale_in : v_scale_in.to(q_scale.scalar_type());
            p.vs_stride_b = v_scale.stride(0); p.vs_stride_h = v_scale.stride(1);
        }
        p.v_scale = v_scale.data_ptr();
    }
    p.batch = (int)Z; p.heads = (int)H; p.seqlen = (int)N; p.head_dim = (int)dk;
    p.heads_kv = (int)Hkv; p.seqlen_k = (int)Nk;
    if (seqlens.defined()) {
        // number of keys per batch entry (a cache filled to different lengths); int32 [Z] on the device
        require_gpu(seqlens);
        if (seqlens.scalar_type() != ScalarType::Int || seqlens.dim() != 1 || seqlens.size(0) != Z)
            fail(PyExc_ValueError, "seqlens_k must be an int32 tensor of shape (" + std::to_string(Z) + ",)");
        seqlens_ = seqlens.contiguous();
        p.seqlens_k = seqlens_.data_ptr<int32_t>();
    }
    // Few queries per head with grouped K/V heads (decoding): the g query heads of a group become g*N rows of ONE head,
    // so that a group streams its K/V once instead of g times.  Pure re-striding: same memory, same results per row.
    // (with the causal mask only where the kernel can be told the position of a row: the decode-shaped calls, which 64-key
    // scale rows under the 128-key block are not)
    const int64_t g = H / Hkv;
    const bool decode_kernel = !(dk == 128 && p.v_scale_block == 64);
    const int64_t fold_rows = !causal ? 2 * kBlockM : (decode_kernel ? kDecodeRows : 0);
    if (g > 1 && g * N <= fold_rows && can_fold(q_, N) && (!scaled || can_fold(q_scale, N))) {
        if (causal) p.causal_rows = (int)N;
        p.heads = p.heads_kv = (int)Hkv; p.seqlen = (int)(g * N);
        p.q_stride_h = g * q_.stride(1); p.q_stride_n = N > 1 ? q_.stride(2) : q_.stride(1);
        p.o_stride_h = g * out.stride(1);
        if (scaled) {
            p.qs_stride_h = g * q_scale.stride(1); p.qs_stride_n = N > 1 ? q_scale.stride(2) : q_scale.stride(1);
        }
    }
    p.io_dtype = io_dtype;
    p.causal = causal ? 1 : 0;
    p.sm_scale = sm_scale;
    p.p_round = p_round;
    if (PyUnicode_Check(a[10])) {
        if (PyUnicode_CompareWithASCIIString(a[10], "auto") != 0) fail(PyExc_ValueError, "num_splits must be a number or \"auto\"");
        p.num_splits = intfa_fwd_suggest_splits(&p, variant, compute_units(dev.device.index()));
        if (p.num_splits < 0) check_rc(p.num_splits, "intfa_fwd_suggest_splits");
    } else {
        p.num_splits = int32_arg(a[10], "num_splits");
    }
    Tensor ws;
    if (p.num_splits > 1) {
        p.workspace_bytes = intfa_fwd_merge_workspace_bytes(&p);
        ws = dev.empty({(int64_t)p.workspace_bytes}, ScalarType::Byte);
        p.workspace = ws.data_ptr();
    }
    void* const st = dev.raw_stream();
    const int rc = unlocked([&] { return full ? intfa_fwd_full_int8(&p, st) : scaled ? intfa_fwd_half_int8(&p, st) : intfa_fwd_fp16(&p, st); });
    check_rc(rc, full ? "intfa_fwd_full_int8" : scaled ? "intfa_fwd_half_int8" : "intfa_fwd_fp16");
    for (const Tensor* t : {&q_, &k_, &v_, &q_scale, const_cast<const Tensor*>(&k_scale), const_cast<const Tensor*>(&v_scale), const_cast<const Tensor*>(&seqlens_)})
        dev.used(*t);
    if (d != dk) out = out.narrow(-1, 0, d).contiguous();
    if (!return_lse) return THPVariable_Wrap(std::move(out));
    PyObject* pair = PyTuple_New(2);
    if (pair == nullptr) throw python_error();
    PyTuple_SET_ITEM(pair, 0, THPVariable_Wrap(std::move(out)));
    PyTuple_SET_ITEM(pair, 1, THPVariable_Wrap(std::move(lse)));
    return pair;
    END_HANDLE_TH_ERRORS
}

// ---- check_head_dims(q, k, v) -> head_dim
PyObject* check_head_dims(PyObject*, PyObject* const* a, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    expect_args(n, 3, "check_head_dims");
    return PyLong_FromLongLong(head_dim_of(tensor_arg(a[0], "q"), tensor_arg(a[1], "k"), tensor_arg(a[2], "v")));
    END_HANDLE_TH_ERRORS
}

// ---- debug_qk_int32(q8, k8): int32 accumulators S = Q8 K8^T as produced by the kernels' MFMA tile code ([Z, H, N, N_k])
PyObject* debug_qk_int32(PyObject*, PyObject* const* a, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    expect_args(n, 2, "debug_qk_int32");
    const Tensor &q = tensor_arg(a[0], "q8"), &k = tensor_arg(a[1], "k8");
    require_gpu(q); require_gpu(k);
    require_4d(q, "q8"); require_4d(k, "k8");
    const int64_t dk = q.size(-1) < kMinHeadDim ? kMinHeadDim : q.size(-1);
    const CallDevice dev(q);
    const Tensor q_ = row_major(q, dk, 1), k_ = row_major(k, dk, 1);
    Tensor s = dev.empty({q.size(0), q.size(1), q.size(2), k.size(2)}, ScalarType::Int);
    intfa_fwd_params p{};
    p.q = q_.data_ptr(); p.k = k_.data_ptr();
    set_strides(&p.q_stride_b, q_); set_strides(&p.k_stride_b, k_);
    p.batch = (int)q.size(0); p.heads = (int)q.size(1); p.seqlen = (int)q.size(2); p.head_dim = (int)dk;
    p.seqlen_k = (int)k.size(2);
    p.scale_dtype = INTFA_F32; p.io_dtype = INTFA_F16;
    void* const st = dev.raw_stream();
    check_rc(unlocked([&] { return intfa_debug_qk_int32(&p, s.data_ptr<int32_t>(), st); }), "intfa_debug_qk_int32");
    dev.used(q_); dev.used(k_);
    return THPVariable_Wrap(std::move(s));
    END_HANDLE_TH_ERRORS
}

// ---- quantisers (benchmark.py:96-107)
int quant_dtype(const Tensor& x) {
    const int t = dtype_enum(x.scalar_type());
    return t == INTFA_F16 || t == INTFA_BF16 ? t : -1;
}
Tensor quant_input(const Tensor& x) {
    if (!x.is_cuda()) fail(PyExc_RuntimeError, "int_flashattention_amd quantisers run on the GPU only; got a CPU tensor");
    if (quant_dtype(x) < 0) fail(PyExc_TypeError, "quantisers take fp16 or bf16 tensors, got " + dtype_text(x.scalar_type()));
    require_4d(x, "x");
    return row_major(x, x.size(-1), 2);
}
PyObject* quant_result(Tensor&& q8, Tensor&& scale) {
    PyObject* pair = PyTuple_New(2);
    if (pair == nullptr) throw python_error();
    PyTuple_SET_ITEM(pair, 0, THPVariable_Wrap(std::move(q8)));
    PyTuple_SET_ITEM(pair, 1, THPVariable_Wrap(std::move(scale)));
    return pair;
}

PyObject* quant_pertoken(PyObject*, PyObject* arg) {
    HANDLE_TH_ERRORS
    const Tensor x = quant_input(tensor_arg(arg, "x"));
    const CallDevice dev(x);
    Tensor q8 = dev.empty(x.sizes(), ScalarType::Char), scale = dev.empty(x.sizes().slice(0, 3), x.scalar_type());
    void* const st = dev.raw_stream();
    const int rc = unlocked([&] {
        return intfa_quant_pertoken(x.data_ptr(), x.stride(0), x.stride(1), x.stride(2), q8.data_ptr(), scale.data_ptr(), (int)x.size(0),
            (int)x.size(1), (int)x.size(2), (int)x.size(3), quant_dtype(x), st);
    });
    check_rc(rc, "intfa_quant_pertoken");
    dev.used(x);
    return quant_result(std::move(q8), std::move(scale));
    END_HANDLE_TH_ERRORS
}

PyObject* quant_pertensor(PyObject*, PyObject* arg) {
    HANDLE_TH_ERRORS
    const Tensor x = quant_input(tensor_arg(arg, "x"));
    const CallDevice dev(x);
    Tensor q8 = dev.empty(x.sizes(), ScalarType::Char), scale = dev.empty(x.sizes().slice(0, 2), x.scalar_type());
    const size_t need = intfa_quant_pertensor_parts_workspace_bytes((int)x.size(0), (int)x.size(1), (int)x.size(2), (int)x.size(3));
    const Tensor ws = dev.empty({(int64_t)need}, ScalarType::Byte);
    void* const st = dev.raw_stream();
    const int rc = unlocked([&] {
        return intfa_quant_pertensor(x.data_ptr(), x.stride(0), x.stride(1), x.stride(2), q8.data_ptr(), scale.data_ptr(), (int)x.size(0),
            (int)x.size(1), (int)x.size(2), (int)x.size(3), quant_dtype(x), ws.data_ptr(), need, st);
    });
    check_rc(rc, "intfa_quant_pertensor");
    dev.used(x);
    return quant_result(std::move(q8), std::move(scale));
    END_HANDLE_TH_ERRORS
}

// quant_perblock_channel(x, block)
PyObject* quant_perblock_channel(PyObject*, PyObject* const* a, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    expect_args(n, 2, "quant_perblock_channel");
    const Tensor x = quant_input(tensor_arg(a[0], "x"));
    const int block = int32_arg(a[1], "block");
    if (block <= 0) fail(PyExc_ValueError, "block must be positive");
    const CallDevice dev(x);
    Tensor q8 = dev.empty(x.sizes(), ScalarType::Char);
    Tensor scale = dev.empty({x.size(0), x.size(1), (x.size(2) + block - 1) / block, x.size(3)}, ScalarType::Float);
    void* const st = dev.raw_stream();
    const int rc = unlocked([&] {
        return intfa_quant_perblock_channel(x.data_ptr(), x.stride(0), x.stride(1), x.stride(2), q8.data_ptr(), scale.data_ptr<float>(),
            (int)x.size(0), (int)x.size(1), (int)x.size(2), (int)x.size(3), block, quant_dtype(x),
            st);
    });
    check_rc(rc, "intfa_quant_perblock_channel");
    dev.used(x);
    return quant_result(std::move(q8), std::move(scale));
    END_HANDLE_TH_ERRORS
}

// ---- kvcache_append(k_cache, k_scale_cache, k_new, seqlens_k, v_cache, v_scale, v_new)
PyObject* kvcache_append(PyObject*, PyObject* const* args, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    expect_args(n, 7, "kvcache_append");
    const Tensor &kc = tensor_arg(args[0], "k_cache"), &ksc = tensor_arg(args[1], "k_scale_cache"), &k_new = tensor_arg(args[2], "k_new");
    const Tensor &vc = optional_tensor_arg(args[4], "v_cache"), &vs = optional_tensor_arg(args[5], "v_scale"), &v_new = optional_tensor_arg(args[6], "v_new");
    if (!kc.is_cuda() || !ksc.is_cuda() || !k_new.is_cuda())
        fail(PyExc_RuntimeError, "int_flashattention_amd.kvcache_append runs on the GPU only; got a CPU tensor");
    if (quant_dtype(k_new) < 0) fail(PyExc_TypeError, "new keys must be fp16 or bf16, got " + dtype_text(k_new.scalar_type()));
    if (kc.scalar_type() != ScalarType::Char || ksc.scalar_type() != k_new.scalar_type())
        fail(PyExc_TypeError, "k_cache must be int8 and k_scale_cache of k_new's dtype");
    require_4d(k_new, "k_new");
    const int64_t Z = k_new.size(0), H = k_new.size(1), Nn = k_new.size(2), d = k_new.size(3);
    if (kc.dim() != 4 || kc.size(0) != Z || kc.size(1) != H || kc.size(3) != d)
        fail(PyExc_ValueError, "k_cache must be [Z, H_kv, N_cache, d] with k_new's Z, H_kv and d");
    const int64_t Nc = kc.size(2);
    if (ksc.dim() != 3 || ksc.size(0) != Z || ksc.size(1) != H || ksc.size(2) != Nc) fail(PyExc_ValueError, "k_scale_cache must be [Z, H_kv, N_cache]");
    if (kc.stride(-1) != 1) fail(PyExc_ValueError, "k_cache rows must be contiguous (the append writes in place)");
    const CallDevice dev(k_new);
    const Tensor kn = quant_input(k_new);
    Tensor vn;
    intfa_append_params a{};
    a.k_new = kn.data_ptr(); set_strides(&a.kn_stride_b, kn);
    a.k_cache = kc.data_ptr(); set_strides(&a.kc_stride_b, kc);
    a.k_scale_cache = ksc.data_ptr(); set_strides(&a.ksc_stride_b, ksc);
    if (v_new.defined()) {
        if (!vc.defined() || !vs.defined()) fail(PyExc_ValueError, "v_new needs v_cache and v_scale");
        if (v_new.scalar_type() != k_new.scalar_type() || vs.scalar_type() != k_new.scalar_type() || vc.scalar_type() != ScalarType::Char)
            fail(PyExc_TypeError, "v_new and v_scale must have k_new's dtype, v_cache must be int8");
        if (v_new.sizes() != k_new.sizes() || vc.sizes() != kc.sizes() || vs.dim() != 2 || vs.size(0) != Z || vs.size(1) != H)
            fail(PyExc_ValueError, "v_new / v_cache / v_scale shapes do not match the keys'");
        if (vc.stride(-1) != 1) fail(PyExc_ValueError, "v_cache rows must be contiguous (the append writes in place)");
        vn = quant_input(v_new);
        a.v_new = vn.data_ptr(); set_strides(&a.vn_stride_b, vn);
        a.v_cache = vc.data_ptr(); set_strides(&a.vc_stride_b, vc);
        a.v_scale = vs.data_ptr(); a.vs_stride_b = vs.stride(0); a.vs_stride_h = vs.stride(1);
    }
    if (PyLong_Check(args[3])) {
        a.seqlen_filled = int32_arg(args[3], "seqlens_k");
    } else {
        const Tensor& len = tensor_arg(args[3], "seqlens_k");
        if (len.scalar_type() != ScalarType::Int || !len.is_cuda() || len.dim() != 1 || len.size(0) != Z || !len.is_contiguous())
            fail(PyExc_ValueError, "seqlens_k must be a contiguous int32 [Z] tensor on the device (or an int)");
        a.seqlens_k = len.data_ptr<int32_t>();
    }
    a.batch = (int)Z; a.heads_kv = (int)H; a.seqlen_new = (int)Nn; a.seqlen_cache = (int)Nc; a.head_dim = (int)d; a.dtype = quant_dtype(k_new);
    void* const st = dev.raw_stream();
    check_rc(unlocked([&] { return intfa_kvcache_append_int8(&a, st); }), "intfa_kvcache_append_int8");
    dev.used(kn); dev.used(vn);
    Py_RETURN_NONE;
    END_HANDLE_TH_ERRORS
}

#define INTFA_FAST(name) {#name, (PyCFunction)(void (*)(void))name, METH_FASTCALL, nullptr}
PyMethodDef methods[] = {
    INTFA_FAST(forward), INTFA_FAST(check_head_dims), INTFA_FAST(debug_qk_int32), INTFA_FAST(quant_perblock_channel), INTFA_FAST(kvcache_append),
    {"quant_pertoken", quant_pertoken, METH_O, nullptr}, {"quant_pertensor", quant_pertensor, METH_O, nullptr},
    {nullptr, nullptr, 0, nullptr}};
PyModuleDef module_def = {PyModuleDef_HEAD_INIT, "_native", "host side of the entry points", -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

extern "C" __attribute__((visibility("default"))) PyObject* PyInit__native(void) {
    if (intfa_version() != INTFA_VERSION) {
        PyErr_Format(PyExc_ImportError, "libintfa.so has ABI version %d, this module expects %d: rebuild it", intfa_version(), INTFA_VERSION);
        return nullptr;
    }
    return PyModule_Create(&module_def);
}
