// The operators' calls in native code: torch tensors in, checked, workspace taken, kernels enqueued.
//
// A decode step's operators run for tens of microseconds on the GPU, and checking twenty to forty tensors in Python
// took as long (fused prolog 43 us of host time per call, attention 14.6): the host, not the GPU, then paces a serving
// loop.  Here a check is a few loads from the tensor object.  Every function takes the operator's arguments by
// position, returns True after enqueueing the kernels, raises what the library reports about a launch -- and returns
// False, with nothing done, for anything it does not take as it is: a wrong type, shape or device, a cache-out that is
// not the cache-in, an unusual scalar.  The Python operator then goes through its own checks, which name the error or
// do the rest (so there is one place that words the errors, and this file need not be complete).
#include "torch_calls.h"

#include <ATen/core/Tensor.h>
#include <c10/core/DeviceGuard.h>
#include <c10/hip/HIPCachingAllocator.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/autograd/python_variable.h>

#include <initializer_list>

#include "pypto_amd_sfa.h"

namespace {

PyTypeObject *wrapper_type = nullptr;      // pypto_amd.converter.Tensor, held for the life of the process
PyObject *wrapper_slot = nullptr;          // the name of its slot that holds the torch tensor

constexpr auto BF16 = at::kBFloat16;
constexpr auto FP16 = at::kHalf;
constexpr auto FP32 = at::kFloat;
constexpr auto I8 = at::kChar;
constexpr auto I32 = at::kInt;
constexpr auto I64 = at::kLong;

// One call's arguments.  Each accessor gives what was asked for, or a harmless value and ok = false.
struct Call {
    PyObject *const *args;
    bool ok = true;
    c10::Device device{c10::DeviceType::CPU, -1};

    const at::Tensor &tensor(const int i)
    {
        static const at::Tensor none;
        PyObject *o = args[i];
        if (Py_TYPE(o) == wrapper_type) {
            o = PyObject_GetAttr(o, wrapper_slot);
            if (o == nullptr) {
                PyErr_Clear();
                ok = false;
                return none;
            }
            Py_DECREF(o);                  // the wrapper keeps it
        }
        if (!THPVariable_Check(o)) {
            ok = false;
            return none;
        }
        const at::Tensor &t = THPVariable_Unpack(o);
        if (t.layout() != c10::kStrided || !t.is_contiguous() || !t.device().is_cuda() || !t.has_storage()) {
            ok = false;
            return none;
        }
        if (device.index() < 0) device = t.device();
        ok = ok && t.device() == device;
        return t;
    }
    // a tensor of a type and, where numel >= 0, a size
    const at::Tensor &of(const int i, const c10::ScalarType type, const int64_t numel = -1)
    {
        const at::Tensor &t = tensor(i);
        ok = ok && t.scalar_type() == type && (numel < 0 || t.numel() == numel);
        return t;
    }
    const at::Tensor &shaped(const int i, const c10::ScalarType type, std::initializer_list<int64_t> sizes)
    {
        const at::Tensor &t = tensor(i);
        ok = ok && t.scalar_type() == type && t.sizes() == c10::IntArrayRef(sizes.begin(), sizes.size());
        return t;
    }
    // the address of a tensor that was checked: ptr for what the kernels read, out for what they write (a tensor that shares
    // its memory copy-on-write gets memory of its own here)
    template <typename T> T *ptr(const at::Tensor &t) { return ok ? static_cast<T *>(const_cast<void *>(t.const_data_ptr())) : nullptr; }
    template <typename T> T *out(const at::Tensor &t) { return ok ? static_cast<T *>(t.mutable_data_ptr()) : nullptr; }

    int64_t integer(const int i)
    {
        if (!PyLong_Check(args[i])) {
            ok = false;
            return 0;
        }
        const int64_t v = PyLong_AsLongLong(args[i]);
        if (v == -1 && PyErr_Occurred()) {
            PyErr_Clear();
            ok = false;
        }
        return v;
    }
    double real(const int i)
    {
        if (!PyFloat_Check(args[i])) {
            ok = false;
            return 0.0;
        }
        return PyFloat_AS_DOUBLE(args[i]);
    }
};

bool dims(const at::Tensor &t, const int64_t n) { return t.defined() && t.dim() == n; }

// a count given as an argument: beyond this the library takes none of them, and the products below stay far from 64 bits
bool count_ok(const int64_t v) { return v >= 1 && v <= (1ll << 24); }

PyObject *declined() { Py_RETURN_FALSE; }

PyObject *raise_status(const int rc)
{
    PyErr_SetString(rc == PTO_E_INVALID_ARG ? PyExc_ValueError : PyExc_RuntimeError, pto_last_error());
    return nullptr;
}

// Workspace from torch's caching allocator on the current stream, then the launch on that stream; the block goes back
// to the allocator at once, which is in stream order, as for a tensor that goes out of scope after the call.
template <typename Args, typename Bytes, typename Launch>
PyObject *enqueue(const c10::Device &device, Args &a, Bytes bytes, Launch launch)
{
    c10::DeviceGuard guard(device);
    const hipStream_t stream = c10::hip::getCurrentHIPStream(device.index()).stream();
    size_t need = 0;
    int rc = bytes(&a, &need);
    if (rc != PTO_OK) return raise_status(rc);
    void *ws = need > 0 ? c10::hip::HIPCachingAllocator::raw_alloc_with_stream(need, stream) : nullptr;
    a.workspace = ws;
    a.workspace_bytes = need;
    rc = launch(&a, stream);
    if (ws != nullptr) c10::hip::HIPCachingAllocator::raw_delete(ws);
    if (rc != PTO_OK) return raise_status(rc);
    Py_RETURN_TRUE;
}

// every exception of torch's accessors (a tensor subclass without storage, an allocator that is out of memory) leaves
// the call to the Python path, which meets the same condition and reports it
template <typename F>
PyObject *guarded(F f)
{
    try {
        return f();
    } catch (const std::exception &) {
        return declined();
    }
}

// query_nope, query_rope, key_nope_2d, key_rope_2d, k_nope_scales (or None), topk_indices, block_table, kv_act_seqs,
// attention_out, nq, n_kv, softmax_scale, topk, block_size, max_blocknum_perbatch
PyObject *sfa_call(PyObject *, PyObject *const *args, Py_ssize_t n)
{
    if (n != 15) return declined();
    return guarded([&]() -> PyObject * {
        Call c{args};
        PtoSfaQuantArgs a{};
        a.nq = c.integer(9), a.n_kv = c.integer(10), a.topk = c.integer(12), a.block_size = c.integer(13);
        const int64_t maxblk = c.integer(14);
        a.softmax_scale = static_cast<float>(c.real(11));
        const at::Tensor &qn = c.of(0, BF16), &kn = c.tensor(2), &bt = c.of(6, I32), &act = c.of(7, I32);
        if (!c.ok || !dims(qn, 2) || !dims(kn, 2) || !dims(bt, 2) || !dims(act, 1) || !count_ok(a.nq) || !count_ok(a.n_kv) || !count_ok(a.topk)) return declined();
        const bool quant = kn.scalar_type() == I8;
        a.b = act.size(0), a.kv_rows = kn.size(0);
        if (a.b < 1 || qn.size(1) != 512 || kn.size(1) != 512 || (!quant && kn.scalar_type() != BF16) || qn.size(0) % (a.b * a.nq) != 0 ||
            bt.size(0) != a.b || bt.size(1) < maxblk || (!quant && args[4] != Py_None))
            return declined();
        a.s1 = qn.size(0) / (a.b * a.nq), a.max_blocknum_perbatch = bt.size(1);
        const at::Tensor &qr = c.shaped(1, BF16, {qn.size(0), 64}), &kr = c.shaped(3, BF16, {a.kv_rows, 64});
        const at::Tensor &ti = c.shaped(5, I32, {a.b * a.s1, a.n_kv * a.topk}), &out = c.shaped(8, BF16, {a.b, a.s1, a.nq, 512});
        if (quant) a.k_nope_scales = c.ptr<void>(c.shaped(4, FP32, {a.kv_rows, 4}));
        if (!c.ok) return declined();
        a.query_nope = c.ptr<void>(qn), a.query_rope = c.ptr<void>(qr), a.key_nope_2d = c.ptr<void>(kn), a.key_rope_2d = c.ptr<void>(kr);
        a.topk_indices = c.ptr<int32_t>(ti), a.block_table = c.ptr<int32_t>(bt), a.kv_act_seqs = c.ptr<int32_t>(act);
        a.attention_out = c.out<void>(out);
        return enqueue(c.device, a, pto_sfa_quant_workspace_bytes, quant ? pto_sfa_quant_launch : pto_sfa_bf16kv_launch);
    });
}

// query_nope, query_rope, nope_cache, topk_indices, block_table, kv_act_seqs, attention_out, nq, n_kv, softmax_scale,
// topk, block_size, max_blocknum_perbatch
PyObject *sa_antiquant_call(PyObject *, PyObject *const *args, Py_ssize_t n)
{
    if (n != 13) return declined();
    return guarded([&]() -> PyObject * {
        Call c{args};
        PtoSaAntiquantArgs a{};
        a.nq = c.integer(7), a.n_kv = c.integer(8), a.topk = c.integer(10), a.block_size = c.integer(11);
        const int64_t maxblk = c.integer(12);
        a.softmax_scale = static_cast<float>(c.real(9));
        const at::Tensor &qn = c.of(0, BF16), &nc = c.of(2, I8), &bt = c.of(4, I32), &act = c.of(5, I32);
        if (!c.ok || !dims(qn, 2) || !dims(nc, 2) || !dims(bt, 2) || !dims(act, 1) || !count_ok(a.nq) || !count_ok(a.n_kv) || !count_ok(a.topk)) return declined();
        a.b = act.size(0), a.kv_rows = nc.size(0);
        if (a.b < 1 || qn.size(1) != 512 || nc.size(1) != 656 || qn.size(0) % (a.b * a.nq) != 0 || bt.size(0) != a.b || bt.size(1) < maxblk)
            return declined();
        a.s1 = qn.size(0) / (a.b * a.nq), a.max_blocknum_perbatch = bt.size(1);
        const at::Tensor &qr = c.shaped(1, BF16, {qn.size(0), 64}), &ti = c.shaped(3, I32, {a.b * a.s1, a.n_kv * a.topk});
        const at::Tensor &out = c.shaped(6, BF16, {a.b, a.s1, a.nq, 512});
        if (!c.ok) return declined();
        a.query_nope = c.ptr<void>(qn), a.query_rope = c.ptr<void>(qr), a.nope_cache = c.ptr<void>(nc);
        a.topk_indices = c.ptr<int32_t>(ti), a.block_table = c.ptr<int32_t>(bt), a.kv_act_seqs = c.ptr<int32_t>(act);
        a.attention_out = c.out<void>(out);
        return enqueue(c.device, a, pto_sa_antiquant_workspace_bytes, pto_sa_antiquant_launch);
    });
}

int dtype_code(const at::Tensor &t, bool &ok)
{
    switch (t.scalar_type()) {
    case FP16: return PTO_DT_FP16;
    case FP32: return PTO_DT_FP32;
    case BF16: return PTO_DT_BF16;
    default: ok = false; return 0;
    }
}

// idx_query, idx_query_scale, idx_key_cache, idx_key_scale, idx_weight, act_seq_key, block_table, topk_res,
// selected_count, arith_variant (0 or 1), most query tokens per sequence, most positions a block table spans
PyObject *li_decode_call(PyObject *, PyObject *const *args, Py_ssize_t n)
{
    if (n != 12) return declined();
    return guarded([&]() -> PyObject * {
        Call c{args};
        PtoLiDecodeArgs a{};
        a.selected_count = c.integer(8), a.arith_variant = static_cast<int32_t>(c.integer(9));
        const int64_t max_s1 = c.integer(10), max_s2 = c.integer(11);
        const at::Tensor &q = c.of(0, I8), &kc = c.of(2, I8), &act = c.of(5, I32), &bt = c.of(6, I32);
        if (!c.ok || !dims(q, 3) || !dims(kc, 4) || !dims(act, 1) || !dims(bt, 2)) return declined();
        a.t = q.size(0), a.n_heads = q.size(1), a.head_dim = q.size(2), a.b = act.size(0);
        a.block_num = kc.size(0), a.block_size = kc.size(1), a.max_blocknum_perbatch = bt.size(1);
        if (a.b < 1 || kc.size(2) != 1 || kc.size(3) != a.head_dim || a.t % a.b != 0 || a.t / a.b > max_s1 || bt.size(0) != a.b ||
            a.max_blocknum_perbatch * a.block_size > max_s2 || !count_ok(a.selected_count))
            return declined();
        const at::Tensor &qs = c.tensor(1), &ks = c.tensor(3), &w = c.tensor(4), &res = c.of(7, I32, a.t * a.selected_count);
        if (!c.ok || qs.numel() != a.t * a.n_heads || w.numel() != a.t * a.n_heads || ks.numel() != a.block_num * a.block_size) return declined();
        a.q_scale_dtype = dtype_code(qs, c.ok), a.k_scale_dtype = dtype_code(ks, c.ok), a.weight_dtype = dtype_code(w, c.ok);
        if (!c.ok || (a.arith_variant != 0 && (qs.scalar_type() != FP16 || ks.scalar_type() != FP16 || w.scalar_type() != FP16))) return declined();
        a.idx_query = c.ptr<int8_t>(q), a.idx_query_scale = c.ptr<void>(qs), a.idx_key_cache = c.ptr<int8_t>(kc), a.idx_key_scale = c.ptr<void>(ks);
        a.idx_weight = c.ptr<void>(w), a.act_seq_key = c.ptr<int32_t>(act), a.block_table = c.ptr<int32_t>(bt), a.topk_res = c.out<int32_t>(res);
        return enqueue(c.device, a, pto_li_decode_workspace_bytes, pto_li_decode_launch);
    });
}

// The two prologs' tensors.  `at` gives the position of each in the call's arguments; the caches appear twice (in and
// out) and have to be the same memory.
bool same_memory(Call &c, const at::Tensor &in, const at::Tensor &out)
{
    return c.ok && in.scalar_type() == out.scalar_type() && in.numel() == out.numel() && c.out<void>(out) == in.const_data_ptr();
}

// at: token_x, w_dq, w_uq_qr, dequant_scale, w_uk, w_dkv_kr, gamma_cq, gamma_ckv, cos, sin, cache_index, kv_cache,
// kr_cache, k_scale_cache, q_norm_out, q_norm_scale_out (both -1: none), query_nope_out, query_rope_out, kv_cache_out,
// kr_cache_out, k_scale_cache_out
bool mla_args(Call &c, const int (&at)[21], PtoMlaPrologQuantArgs &a)
{
    const at::Tensor &x = c.of(at[0], BF16), &wdq = c.of(at[1], BF16), &wuk = c.of(at[4], BF16), &kvc = c.of(at[18], I8);
    if (!c.ok || !dims(x, 2) || !dims(wdq, 2) || !dims(wuk, 3) || !dims(kvc, 4)) return false;
    a.t = x.size(0), a.h = x.size(1), a.q_lora_rank = wdq.size(1), a.n_heads = wuk.size(0), a.cache_rows = kvc.size(0) * kvc.size(1);
    const at::Tensor &krc = c.of(at[19], BF16, a.cache_rows * 64), &ksc = c.of(at[20], FP32, a.cache_rows * 4);
    if (!c.ok || !dims(krc, 4) || wdq.size(0) != a.h || wuk.size(1) != 128 || wuk.size(2) != 512 || kvc.size(2) != 1 || kvc.size(3) != 512 ||
        krc.size(2) != 1 || krc.size(3) != 64)
        return false;
    if (!same_memory(c, c.tensor(at[11]), kvc) || !same_memory(c, c.tensor(at[12]), krc) || !same_memory(c, c.tensor(at[13]), ksc)) return false;
    a.token_x = c.ptr<void>(x), a.w_dq = c.ptr<void>(wdq), a.w_uk = c.ptr<void>(wuk);
    a.kv_cache = c.out<int8_t>(kvc), a.kr_cache = c.out<void>(krc), a.k_scale_cache = c.out<float>(ksc);
    a.w_uq_qr = c.ptr<int8_t>(c.shaped(at[2], I8, {a.q_lora_rank, a.n_heads * 192}));
    a.dequant_scale = c.ptr<float>(c.of(at[3], FP32, a.n_heads * 192));
    a.w_dkv_kr = c.ptr<void>(c.shaped(at[5], BF16, {a.h, 576}));
    a.gamma_cq = c.ptr<void>(c.of(at[6], BF16, a.q_lora_rank));
    a.gamma_ckv = c.ptr<void>(c.of(at[7], BF16, 512));
    a.cos = c.ptr<void>(c.of(at[8], BF16, a.t * 64));
    a.sin = c.ptr<void>(c.of(at[9], BF16, a.t * 64));
    a.cache_index = c.ptr<int64_t>(c.of(at[10], I64, a.t));
    if (at[14] >= 0) {
        a.q_norm_out = c.out<int8_t>(c.of(at[14], I8, a.t * a.q_lora_rank));
        a.q_norm_scale_out = c.out<float>(c.of(at[15], FP32, a.t));
    }
    a.query_nope_out = c.out<void>(c.of(at[16], BF16, a.t * a.n_heads * 512));
    a.query_rope_out = c.out<void>(c.of(at[17], BF16, a.t * a.n_heads * 64));
    return c.ok;
}

// at: x, q_norm, q_norm_scale (both -1: made by the MLA half), w_qb, w_qb_scale, wk, w_proj, ln_gamma_k, ln_beta_k, cos,
// sin, hadamard_q, hadamard_k, k_int8, k_scale, k_cache_index, q_int8_out, q_scale_out, k_int8_out, k_scale_out, weights_out
bool li_prolog_args(Call &c, const int (&at)[21], PtoLiPrologQuantArgs &a)
{
    const at::Tensor &x = c.of(at[0], BF16), &wqb = c.of(at[3], I8), &wp = c.of(at[6], BF16), &kc = c.of(at[18], I8);
    const at::Tensor &cos = c.tensor(at[9]), &sin = c.tensor(at[10]);
    if (!c.ok || !dims(x, 2) || !dims(wqb, 2) || !dims(wp, 2) || !dims(kc, 4) || cos.dim() < 1 || sin.dim() < 1) return false;
    a.t = x.size(0), a.h = x.size(1), a.q_lora_rank = wqb.size(0), a.n_heads = wp.size(1), a.cache_rows = kc.size(0) * kc.size(1);
    const at::Tensor &ks = c.of(at[19], FP16, a.cache_rows);
    if (!c.ok || wp.size(0) != a.h || wqb.size(1) != a.n_heads * 128 || kc.size(2) != 1 || kc.size(3) != 128 || cos.size(-1) != 64 || sin.size(-1) != 64)
        return false;
    const at::Tensor &kc_in = c.of(at[13], I8);
    if (!same_memory(c, kc_in, kc) || kc_in.sizes() != kc.sizes() || !same_memory(c, c.tensor(at[14]), ks)) return false;
    a.x = c.ptr<void>(x), a.w_qb = c.ptr<int8_t>(wqb), a.w_proj = c.ptr<void>(wp), a.k_cache = c.out<int8_t>(kc), a.k_cache_scale = c.out<void>(ks);
    if (at[1] >= 0) {
        a.q_norm = c.ptr<int8_t>(c.shaped(at[1], I8, {a.t, a.q_lora_rank}));
        a.q_norm_scale = c.ptr<float>(c.of(at[2], FP32, a.t));
    }
    a.w_qb_scale = c.ptr<float>(c.of(at[4], FP32, a.n_heads * 128));
    a.wk = c.ptr<void>(c.shaped(at[5], BF16, {a.h, 128}));
    a.ln_gamma_k = c.ptr<void>(c.of(at[7], BF16, 128));
    a.ln_beta_k = c.ptr<void>(c.of(at[8], BF16, 128));
    a.cos_idx_rope = c.ptr<void>(c.of(at[9], BF16, a.t * 64));
    a.sin_idx_rope = c.ptr<void>(c.of(at[10], BF16, a.t * 64));
    a.hadamard_q = c.ptr<void>(c.shaped(at[11], BF16, {128, 128}));
    a.hadamard_k = c.ptr<void>(c.shaped(at[12], BF16, {128, 128}));
    a.k_cache_index = c.ptr<int64_t>(c.of(at[15], I64, a.t));
    a.q_int8 = c.out<int8_t>(c.of(at[16], I8, a.t * a.n_heads * 128));
    a.q_scale = c.out<void>(c.of(at[17], FP16, a.t * a.n_heads));
    a.weights = c.out<void>(c.of(at[20], FP16, a.t * a.n_heads));
    return c.ok;
}

// the operator's 21 tensors, epsilon_cq, epsilon_ckv, absorb_exact
PyObject *mla_prolog_call(PyObject *, PyObject *const *args, Py_ssize_t n)
{
    if (n != 24) return declined();
    return guarded([&]() -> PyObject * {
        Call c{args};
        PtoMlaPrologQuantArgs a{};
        static constexpr int at[21] = {0, 1, 2, 3, 4, 5, 6, 7, 8, 9, 10, 11, 12, 13, 14, 15, 16, 17, 18, 19, 20};
        a.epsilon_cq = static_cast<float>(c.real(21)), a.epsilon_ckv = static_cast<float>(c.real(22));
        a.absorb_exact = args[23] == Py_True ? 1 : 0;
        if (!mla_args(c, at, a)) return declined();
        return enqueue(c.device, a, pto_mla_prolog_quant_workspace_bytes, pto_mla_prolog_quant_launch);
    });
}

// the operator's 21 tensors, eps, sum_mode
PyObject *li_prolog_call(PyObject *, PyObject *const *args, Py_ssize_t n)
{
    if (n != 23) return declined();
    return guarded([&]() -> PyObject * {
        Call c{args};
        PtoLiPrologQuantArgs a{};
        static constexpr int at[21] = {0, 1, 2, 3, 4, 5, 6, 7, 8, 9, 10, 11, 12, 13, 14, 15, 16, 17, 18, 19, 20};
        a.eps = static_cast<float>(c.real(21)), a.sum_mode = static_cast<int32_t>(c.integer(22));
        if (!li_prolog_args(c, at, a)) return declined();
        return enqueue(c.device, a, pto_li_prolog_quant_workspace_bytes, pto_li_prolog_quant_launch);
    });
}

// the operator's 34 tensors, epsilon_cq, epsilon_ckv, absorb_exact, eps, sum_mode
PyObject *fused_prolog_call(PyObject *, PyObject *const *args, Py_ssize_t n)
{
    if (n != 39) return declined();
    return guarded([&]() -> PyObject * {
        Call c{args};
        PtoMlaIndexerPrologQuantArgs a{};
        static constexpr int mla[21] = {0, 1, 2, 3, 4, 5, 6, 7, 8, 9, 10, 11, 12, 13, -1, -1, 24, 25, 26, 27, 28};
        static constexpr int idx[21] = {0, -1, -1, 14, 15, 16, 17, 18, 19, 8, 9, 20, 21, 22, 23, 10, 29, 30, 31, 32, 33};
        a.mla.epsilon_cq = static_cast<float>(c.real(34)), a.mla.epsilon_ckv = static_cast<float>(c.real(35));
        a.mla.absorb_exact = args[36] == Py_True ? 1 : 0;
        a.indexer.eps = static_cast<float>(c.real(37)), a.indexer.sum_mode = static_cast<int32_t>(c.integer(38));
        if (!mla_args(c, mla, a.mla) || !li_prolog_args(c, idx, a.indexer) || a.mla.q_lora_rank != a.indexer.q_lora_rank) return declined();
        return enqueue(c.device, a, pto_mla_indexer_prolog_quant_workspace_bytes, pto_mla_indexer_prolog_quant_launch);
    });
}

// the wrapper class whose instances stand for their torch tensor, and the name of the slot that holds it
PyObject *set_wrapper(PyObject *, PyObject *const *args, Py_ssize_t n)
{
    if (n != 2 || !PyType_Check(args[0]) || !PyUnicode_Check(args[1])) {
        PyErr_SetString(PyExc_TypeError, "set_wrapper: a type and the name of its slot");
        return nullptr;
    }
    Py_INCREF(args[0]);
    Py_INCREF(args[1]);
    Py_XDECREF(reinterpret_cast<PyObject *>(wrapper_type));
    Py_XDECREF(wrapper_slot);
    wrapper_type = reinterpret_cast<PyTypeObject *>(args[0]);
    wrapper_slot = args[1];
    Py_RETURN_NONE;
}

#define FAST(name) {#name, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)(void)>(name)), METH_FASTCALL, nullptr}
PyMethodDef methods[] = {FAST(sfa_call),       FAST(sa_antiquant_call), FAST(li_decode_call), FAST(mla_prolog_call),
                         FAST(li_prolog_call), FAST(fused_prolog_call), FAST(set_wrapper),    {nullptr, nullptr, 0, nullptr}};
#undef FAST

}  // namespace

int pto::add_torch_calls(PyObject *module) { return PyModule_AddFunctions(module, methods); }
