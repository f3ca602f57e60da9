// Thin PyTorch-ROCm glue: the pybind module `attnkernels_ext` with the
// reference's four functions (attnkernels/csrc/ext.cpp:3-17) plus the paged
// cache writer reshape_and_cache and the GQA / varlen prefill, each allocating
// its output (and split-K workspace) from the caching allocator and calling
// the C-ABI in include/attnkernels.h on the caller's current HIP stream.
#include <torch/extension.h>

// PyTorch-ROCm reports GPU tensors with device type "cuda"; these are its
// guard and stream accessors for that device type.
#include <ATen/hip/impl/HIPGuardImplMasqueradingAsCUDA.h>
#include <ATen/hip/impl/HIPStreamMasqueradingAsCUDA.h>

#include <algorithm>
#include <cmath>
#include <map>
#include <mutex>
#include <utility>
#include <vector>

#include "attnkernels.h"

namespace {

void check_rc(int rc) { TORCH_CHECK(rc == AK_OK, ak_last_error()); }

void check_prefill(const torch::Tensor& q, const torch::Tensor& k, const torch::Tensor& v) {
    for (const auto* t : {&q, &k, &v}) {
        TORCH_CHECK(t->is_cuda() && t->scalar_type() == torch::kHalf && t->dim() == 4 && t->is_contiguous(),
                    "q, k, v must be contiguous fp16 GPU tensors of shape [B, H, N, D]");
        TORCH_CHECK(t->device() == q.device(), "q, k, v must be on the same device");
    }
    TORCH_CHECK(q.sizes() == k.sizes() && q.sizes() == v.sizes(),
                "q, k, v must have the same shape (self-attention prefill)");
}

void* stream_of(const torch::Tensor& t) {
    return at::hip::getCurrentHIPStreamMasqueradingAsCUDA(t.device().index()).stream();
}

// The stream capture that calls on `stream` are recorded into, 0: none.
unsigned long long capture_id(void* stream) {
    hipStreamCaptureStatus status = hipStreamCaptureStatusNone;
    unsigned long long id = 0;
    if (hipStreamGetCaptureInfo(static_cast<hipStream_t>(stream), &status, &id) != hipSuccess) return 0;
    return status == hipStreamCaptureStatusNone ? 0 : id;
}

// Split counters of the decode kernels' in-kernel merge, one array per
// (device, stream): zeroed when allocated, and every decode call leaves its
// counters at zero, so the calls on a stream (which run in order) share it.
// The calls recorded into a graph share another one, per stream and capture:
// what zeroes it is recorded before them, so each replay starts from zeros
// whatever has used that memory since (graphs that share a memory pool reuse
// each other's), and two graphs never share counters.  It is let go when the
// stream records the next graph; an array grown during a capture is kept that long too.
// The cache is never destroyed: its tensors would otherwise be freed during
// static destruction, after torch's allocator or the HIP runtime may be gone.
torch::Tensor split_counters(const torch::Tensor& q, int64_t n) {
    struct Arrays {
        torch::Tensor eager;
        unsigned long long capture = 0;
        std::vector<torch::Tensor> captured;
    };
    static std::mutex mu;
    static auto* cache = new std::map<std::pair<int, void*>, Arrays>();
    void* const stream = stream_of(q);
    const unsigned long long capture = capture_id(stream);
    std::lock_guard<std::mutex> lock(mu);
    auto& arrays = (*cache)[{(int)q.device().index(), stream}];
    if (capture != 0 && arrays.capture != capture) {
        arrays.captured.clear();
        arrays.capture = capture;
    }
    torch::Tensor last = capture == 0                ? arrays.eager
                         : arrays.captured.empty() ? torch::Tensor()
                                                     : arrays.captured.back();
    if (!last.defined() || last.numel() < n) {
        const int64_t grow = last.defined() ? 2 * last.numel() : 0;
        last = torch::zeros({std::max(n, std::max<int64_t>(grow, 4096))}, q.options().dtype(torch::kInt));
        if (capture == 0) arrays.eager = last;
        else arrays.captured.push_back(last);
    }
    return last;
}

}  // namespace

torch::Tensor naive_attention(const torch::Tensor& q, const torch::Tensor& k, const torch::Tensor& v, bool causal, double scale) {
    check_prefill(q, k, v);
    const at::hip::HIPGuardMasqueradingAsCUDA guard(q.device());
    auto o = torch::empty_like(q);
    check_rc(ak_naive_attention(q.data_ptr(), k.data_ptr(), v.data_ptr(), o.data_ptr(), q.size(0), q.size(1),
                                q.size(2), q.size(3), causal, scale, stream_of(q)));
    return o;
}

torch::Tensor flash_simt(const torch::Tensor& q, const torch::Tensor& k, const torch::Tensor& v, bool causal, double scale) {
    check_prefill(q, k, v);
    const at::hip::HIPGuardMasqueradingAsCUDA guard(q.device());
    auto o = torch::empty_like(q);
    check_rc(ak_flash_simt(q.data_ptr(), k.data_ptr(), v.data_ptr(), o.data_ptr(), q.size(0), q.size(1),
                           q.size(2), q.size(3), causal, scale, stream_of(q)));
    return o;
}

torch::Tensor flash_wmma(const torch::Tensor& q, const torch::Tensor& k, const torch::Tensor& v, bool causal, double scale,
                         int64_t block_n) {
    check_prefill(q, k, v);
    const at::hip::HIPGuardMasqueradingAsCUDA guard(q.device());
    auto o = torch::empty_like(q);
    check_rc(ak_flash_wmma(q.data_ptr(), k.data_ptr(), v.data_ptr(), o.data_ptr(), q.size(0), q.size(1),
                           q.size(2), q.size(3), causal, scale, block_n, stream_of(q)));
    return o;
}

// Dense prefill with fewer kv heads than query heads (GQA/MQA).
torch::Tensor flash_gqa(const torch::Tensor& q, const torch::Tensor& k, const torch::Tensor& v, bool causal, double scale) {
    for (const auto* t : {&q, &k, &v}) {
        TORCH_CHECK(t->is_cuda() && t->scalar_type() == torch::kHalf && t->dim() == 4 && t->is_contiguous(),
                    "q, k, v must be contiguous fp16 GPU tensors of shape [B, H, N, D]");
        TORCH_CHECK(t->device() == q.device(), "q, k, v must be on the same device");
    }
    TORCH_CHECK(k.sizes() == v.sizes() && k.size(0) == q.size(0) && k.size(2) == q.size(2) && k.size(3) == q.size(3),
                "k and v must be [B, H_kv, N, D] with q's B, N and D");
    const at::hip::HIPGuardMasqueradingAsCUDA guard(q.device());
    auto o = torch::empty_like(q);
    check_rc(ak_prefill_gqa(q.data_ptr(), k.data_ptr(), v.data_ptr(), o.data_ptr(), q.size(0), q.size(1), k.size(1),
                            q.size(2), q.size(3), causal, scale, stream_of(q)));
    return o;
}

// Packed variable-length prefill: q [T, H, D], k/v [T, H_kv, D], cu_seqlens int32 [B + 1].
torch::Tensor flash_varlen(const torch::Tensor& q, const torch::Tensor& k, const torch::Tensor& v, const torch::Tensor& cu, int64_t max_seqlen,
                           bool causal, double scale) {
    for (const auto* t : {&q, &k, &v}) {
        TORCH_CHECK(t->is_cuda() && t->scalar_type() == torch::kHalf && t->dim() == 3 && t->is_contiguous(),
                    "q, k, v must be contiguous fp16 GPU tensors of shape [total, H, D]");
        TORCH_CHECK(t->device() == q.device(), "q, k, v must be on the same device");
    }
    TORCH_CHECK(k.sizes() == v.sizes() && k.size(0) == q.size(0) && k.size(2) == q.size(2),
                "k and v must be [total, H_kv, D] with q's total and D");
    TORCH_CHECK(cu.scalar_type() == torch::kInt && cu.dim() == 1 && cu.is_contiguous() && cu.size(0) >= 1 &&
                    cu.device() == q.device(),
                "cu_seqlens must be a contiguous int32 tensor [B + 1] on q's device");
    const at::hip::HIPGuardMasqueradingAsCUDA guard(q.device());
    auto o = torch::empty_like(q);
    check_rc(ak_prefill_varlen(q.data_ptr(), k.data_ptr(), v.data_ptr(), o.data_ptr(), cu.data_ptr<int32_t>(),
                               cu.size(0) - 1, q.size(0), q.size(1), k.size(1), max_seqlen, q.size(2), causal, scale,
                               stream_of(q)));
    return o;
}

// balanced: splits cut by the kernel from the context lengths, where they serve.
static torch::Tensor decode(const torch::Tensor& q, const torch::Tensor& kc, const torch::Tensor& vc,
                            const torch::Tensor& bt, const torch::Tensor& ctx, int64_t max_ctx, double scale,
                            int64_t partition, bool balanced) {
    TORCH_CHECK(q.is_cuda() && q.scalar_type() == torch::kHalf && q.dim() == 3 && q.is_contiguous(),
                "q must be a contiguous fp16 GPU tensor [B, H, D]");
    TORCH_CHECK(kc.is_cuda() && kc.scalar_type() == torch::kHalf && kc.dim() == 4 && kc.is_contiguous() &&
                    vc.sizes() == kc.sizes() && vc.scalar_type() == torch::kHalf && vc.is_contiguous(),
                "k_cache and v_cache must be contiguous fp16 GPU tensors [num_blocks, H_kv, block_size, D]");
    TORCH_CHECK(kc.size(3) == q.size(2), "head_dim of q and the cache must match");
    TORCH_CHECK(bt.scalar_type() == torch::kInt && bt.dim() == 2 && bt.is_contiguous() && bt.size(0) == q.size(0),
                "block_tables must be a contiguous int32 tensor [B, max_blocks]");
    TORCH_CHECK(ctx.scalar_type() == torch::kInt && ctx.dim() == 1 && ctx.is_contiguous() && ctx.size(0) == q.size(0),
                "context_lens must be a contiguous int32 tensor [B]");
    for (const auto* t : {&kc, &vc, &bt, &ctx})
        TORCH_CHECK(t->device() == q.device(), "all paged_decode tensors must be on the same device");
    const at::hip::HIPGuardMasqueradingAsCUDA guard(q.device());
    auto out = torch::empty_like(q);
    const int64_t B = q.size(0), hq = q.size(1), D = q.size(2), hkv = kc.size(1);
    size_t ws_bytes = balanced ? ak_paged_decode_balanced_workspace_size(B, hq, hkv, D, max_ctx, partition) : 0;
    const auto run = ws_bytes > 0 ? ak_paged_decode_balanced : ak_paged_decode_fused;
    if (ws_bytes == 0) ws_bytes = ak_paged_decode_workspace_size(B, hq, D, max_ctx, partition);
    torch::Tensor ws, counters;
    if (ws_bytes > 0) {
        ws = torch::empty({(int64_t)ws_bytes}, q.options().dtype(torch::kByte));
        counters = split_counters(q, B * hkv);
    }
    check_rc(run(q.data_ptr(), kc.data_ptr(), vc.data_ptr(), bt.data_ptr<int32_t>(), ctx.data_ptr<int32_t>(),
                 out.data_ptr(), B, hq, hkv, D, kc.size(0), kc.size(2), bt.size(1), max_ctx, scale, partition,
                 ws_bytes ? ws.data_ptr() : nullptr, ws_bytes, ws_bytes ? counters.data_ptr<int32_t>() : nullptr,
                 ws_bytes ? counters.numel() : 0, stream_of(q)));
    return out;
}

torch::Tensor paged_decode(torch::Tensor q, torch::Tensor kc, torch::Tensor vc, torch::Tensor bt,
                           torch::Tensor ctx, int64_t max_ctx, double scale, int64_t partition) {
    return decode(q, kc, vc, bt, ctx, max_ctx, scale, partition, false);
}

// Splits of about equal size where they serve, else of `partition` tokens.
torch::Tensor paged_decode_balanced(torch::Tensor q, torch::Tensor kc, torch::Tensor vc, torch::Tensor bt,
                                    torch::Tensor ctx, int64_t max_ctx, double scale, int64_t partition) {
    return decode(q, kc, vc, bt, ctx, max_ctx, scale, partition, true);
}

// In place: writes key/value rows into the caches (no counterpart in the
// reference, whose decode only reads the cache).
void reshape_and_cache(const torch::Tensor& key, const torch::Tensor& value, const torch::Tensor& kc,
                       const torch::Tensor& vc, const torch::Tensor& slots) {
    TORCH_CHECK(key.is_cuda() && key.dim() == 3 && value.dim() == 3 && key.sizes() == value.sizes(),
                "key and value must be GPU tensors [num_tokens, H_kv, D] of the same shape");
    TORCH_CHECK(key.element_size() == 2 && value.scalar_type() == key.scalar_type() &&
                    kc.scalar_type() == key.scalar_type() && vc.scalar_type() == key.scalar_type(),
                "key, value and the caches must share one 2-byte dtype (fp16 or bf16)");
    TORCH_CHECK(key.stride(2) == 1 && key.stride(1) == key.size(2) && value.stride(2) == 1 &&
                    value.stride(1) == value.size(2),
                "key and value must have contiguous heads (any token stride)");
    TORCH_CHECK(kc.dim() == 4 && kc.is_contiguous() && vc.is_contiguous() && vc.sizes() == kc.sizes() &&
                    kc.size(1) == key.size(1) && kc.size(3) == key.size(2),
                "k_cache and v_cache must be contiguous [num_blocks, H_kv, block_size, D] matching key");
    TORCH_CHECK(slots.scalar_type() == torch::kLong && slots.dim() == 1 && slots.is_contiguous() &&
                    slots.size(0) == key.size(0),
                "slot_mapping must be a contiguous int64 tensor [num_tokens]");
    for (const auto* t : {&value, &kc, &vc, &slots})
        TORCH_CHECK(t->device() == key.device(), "all reshape_and_cache tensors must be on the same device");
    const at::hip::HIPGuardMasqueradingAsCUDA guard(key.device());
    const int64_t T = key.size(0);
    check_rc(ak_reshape_and_cache(key.data_ptr(), value.data_ptr(), kc.data_ptr(), vc.data_ptr(),
                                  slots.data_ptr<int64_t>(), T, key.size(1), key.size(2), kc.size(0), kc.size(2),
                                  T > 1 ? key.stride(0) : key.size(1) * key.size(2),
                                  T > 1 ? value.stride(0) : value.size(1) * value.size(2), stream_of(key)));
}

// XOR checksum of a tensor's bytes (a multiple of 16): the read-only
// streaming kernel behind bench.py's HBM read ceiling.
// out (int32[4] on x's device) accumulates the XOR when given: the caller
// zeroes it; without it a zeroed one is made.
torch::Tensor stream_checksum(torch::Tensor x, c10::optional<torch::Tensor> out_opt) {
    TORCH_CHECK(x.is_cuda() && x.is_contiguous() && x.nbytes() % 16 == 0,
                "stream_checksum: a contiguous GPU tensor of a multiple of 16 bytes");
    const at::hip::HIPGuardMasqueradingAsCUDA guard(x.device());
    torch::Tensor out;
    if (out_opt.has_value()) {
        out = *out_opt;
        TORCH_CHECK(out.device() == x.device() && out.scalar_type() == torch::kInt && out.numel() == 4 &&
                        out.is_contiguous(),
                    "stream_checksum: out must be a contiguous int32[4] on the input's device");
    } else {
        out = torch::zeros({4}, x.options().dtype(torch::kInt));
    }
    check_rc(ak_stream_checksum(x.data_ptr(), x.nbytes(), reinterpret_cast<uint32_t*>(out.data_ptr<int32_t>()),
                                stream_of(x)));
    return out;
}

// ---------------------------------------------------------------------------
// The calls the Python wrappers make first.  Each takes the arguments as the
// user gave them and runs the call if they are the plain case (ordinary
// contiguous GPU tensors of the right types and shapes, True/False, ints,
// floats or None); otherwise it returns None, touching nothing, and the
// wrapper checks, converts or refuses them in Python.  The checks here are the
// wrappers' and this file's, in one pass: measured on an MI355X host, a
// 64-token reshape_and_cache call 7.0 -> 3.4 us, the smallest prefill 6.0 ->
// 4.6 us of host time.
namespace {

// o as an ordinary GPU tensor (exactly torch.Tensor, no functorch or
// torch-dispatch wrapper), or null.
const at::Tensor* plain(PyObject* o) {
    if (!THPVariable_CheckExact(o)) return nullptr;
    const at::Tensor& t = THPVariable_Unpack(o);
    constexpr c10::DispatchKeySet wrapped({c10::DispatchKey::Python, c10::DispatchKey::FuncTorchBatched,
                                           c10::DispatchKey::FuncTorchGradWrapper, c10::DispatchKey::Functionalize,
                                           c10::DispatchKey::Conjugate, c10::DispatchKey::Negative});
    if (!t.is_cuda() || t.layout() != c10::kStrided || t.key_set().has_any(wrapped)) return nullptr;
    return &t;
}

bool plain_int(PyObject* o, int64_t& x) {
    if (!PyLong_CheckExact(o)) return false;
    int overflow = 0;
    x = PyLong_AsLongLongAndOverflow(o, &overflow);
    return overflow == 0;
}

// None: 1 / sqrt(head_dim).
bool plain_scale(PyObject* o, int64_t head_dim, double& x) {
    if (o == Py_None) x = 1.0 / std::sqrt((double)head_dim);
    else if (PyFloat_CheckExact(o)) x = PyFloat_AS_DOUBLE(o);
    else return false;
    return true;
}

bool half_tensors(std::initializer_list<const at::Tensor*> ts, int64_t dim) {
    const at::Tensor& first = **ts.begin();
    for (const at::Tensor* t : ts)
        if (t->scalar_type() != at::kHalf || t->dim() != dim || !t->is_contiguous() || t->device() != first.device())
            return false;
    return true;
}

py::object none() { return py::none(); }

}  // namespace

// flash_attention with its default variant (heads equal), flash_attention_gqa (kv heads dividing the heads).
py::object plain_prefill(py::handle qo, py::handle ko, py::handle vo, py::handle causal, py::handle scale, bool gqa) {
    const at::Tensor *q = plain(qo.ptr()), *k = plain(ko.ptr()), *v = plain(vo.ptr());
    if (!q || !k || !v || !PyBool_Check(causal.ptr()) || !half_tensors({q, k, v}, 4) || k->sizes() != v->sizes())
        return none();
    const int64_t D = q->size(3);
    double s;
    if ((D != 64 && D != 128) || !plain_scale(scale.ptr(), D, s)) return none();
    if (gqa ? k->size(0) != q->size(0) || k->size(2) != q->size(2) || k->size(3) != D || k->size(1) == 0 ||
                  q->size(1) % k->size(1) != 0
            : q->sizes() != k->sizes())
        return none();
    const bool c = causal.ptr() == Py_True;
    return py::cast(gqa ? flash_gqa(*q, *k, *v, c, s) : flash_wmma(*q, *k, *v, c, s, 64));
}

py::object plain_varlen(py::handle qo, py::handle ko, py::handle vo, py::handle cuo, py::handle max_seqlen,
                        py::handle causal, py::handle scale) {
    const at::Tensor *q = plain(qo.ptr()), *k = plain(ko.ptr()), *v = plain(vo.ptr()), *cu = plain(cuo.ptr());
    if (!q || !k || !v || !cu || !PyBool_Check(causal.ptr()) || !half_tensors({q, k, v}, 3) || k->sizes() != v->sizes())
        return none();
    const int64_t D = q->size(2);
    double s;
    int64_t longest;
    if ((D != 64 && D != 128) || k->size(0) != q->size(0) || k->size(2) != D || k->size(1) == 0 ||
        q->size(1) % k->size(1) != 0 || !plain_scale(scale.ptr(), D, s) || !plain_int(max_seqlen.ptr(), longest))
        return none();
    if (cu->scalar_type() != at::kInt || cu->dim() != 1 || cu->size(0) < 1 || !cu->is_contiguous() ||
        cu->device() != q->device())
        return none();
    return py::cast(flash_varlen(*q, *k, *v, *cu, longest, causal.ptr() == Py_True, s));
}

// partition(batch, kv heads, max_context_len, device): decode_partition, called when partition_size is None.
py::object plain_decode(py::handle qo, py::handle kco, py::handle vco, py::handle bto, py::handle ctxo,
                        py::handle max_context_len, py::handle scale, py::handle partition_size,
                        py::handle partition) {
    const at::Tensor *q = plain(qo.ptr()), *kc = plain(kco.ptr()), *vc = plain(vco.ptr()), *bt = plain(bto.ptr()),
                     *ctx = plain(ctxo.ptr());
    if (!q || !kc || !vc || !bt || !ctx || !half_tensors({q}, 3) || !half_tensors({kc, vc}, 4)) return none();
    const int64_t D = q->size(2);
    double s;
    int64_t longest, part;
    if ((D != 64 && D != 128) || kc->size(3) != D || kc->sizes() != vc->sizes() || kc->device() != q->device() ||
        !plain_scale(scale.ptr(), D, s) || !plain_int(max_context_len.ptr(), longest))
        return none();
    for (const at::Tensor* t : {bt, ctx})
        if (t->scalar_type() != at::kInt || !t->is_contiguous() || t->device() != q->device() ||
            t->dim() != (t == bt ? 2 : 1) || t->size(0) != q->size(0))
            return none();
    const bool balanced = partition_size.is_none();
    if (balanced) {
        if (q->size(0) == 0 || kc->size(1) == 0 || longest < 1) return none();
        part = partition(q->size(0), kc->size(1), longest, (int64_t)q->device().index()).cast<int64_t>();
    } else {
        if (!plain_int(partition_size.ptr(), part) || part < 1 || part > INT32_MAX) return none();
        part = (part + 255) / 256 * 256;
    }
    return py::cast(decode(*q, *kc, *vc, *bt, *ctx, longest, s, part, balanced));
}

// True if the rows were written.
bool plain_write(py::handle ko, py::handle vo, py::handle kco, py::handle vco, py::handle so) {
    const at::Tensor *key = plain(ko.ptr()), *value = plain(vo.ptr()), *kc = plain(kco.ptr()), *vc = plain(vco.ptr()),
                     *slots = plain(so.ptr());
    if (!key || !value || !kc || !vc || !slots) return false;
    const auto type = key->scalar_type();
    if ((type != at::kHalf && type != at::kBFloat16) || key->dim() != 3 || kc->dim() != 4 ||
        key->sizes() != value->sizes() || kc->sizes() != vc->sizes() || kc->size(1) != key->size(1) ||
        kc->size(3) != key->size(2) || key->size(2) % 8 != 0 || key->size(0) < 1)
        return false;
    for (const at::Tensor* t : {value, kc, vc})
        if (t->scalar_type() != type || t->device() != key->device()) return false;
    for (const at::Tensor* t : {key, value})  // heads contiguous, token stride and start on 16 bytes
        if (t->stride(2) != 1 || t->stride(1) != t->size(2) || (t->size(0) > 1 && t->stride(0) % 8 != 0) ||
            reinterpret_cast<uintptr_t>(t->data_ptr()) % 16 != 0)
            return false;
    if (!kc->is_contiguous() || !vc->is_contiguous() || slots->scalar_type() != at::kLong || slots->dim() != 1 ||
        slots->size(0) != key->size(0) || !slots->is_contiguous() || slots->device() != key->device())
        return false;
    reshape_and_cache(*key, *value, *kc, *vc, *slots);
    return true;
}

PYBIND11_MODULE(TORCH_EXTENSION_NAME, m) {
    m.doc() = "gfx950 attention kernels: MFMA flash prefill, paged split-K decode";
    m.def("naive_attention", &naive_attention, "prefill attention (served by the MFMA flash kernel)");
    m.def("flash_simt", &flash_simt, "prefill attention (served by the MFMA flash kernel)");
    m.def("flash_wmma", &flash_wmma, "tiled attention with online softmax on MFMA matrix cores");
    m.def("paged_decode", &paged_decode, "decode attention over a paged KV cache, split-K");
    m.def("paged_decode_balanced", &paged_decode_balanced, "the same with splits cut evenly over the batch's contexts");
    m.def("stream_checksum", &stream_checksum, "XOR checksum of a tensor's bytes (read-only streaming ceiling)",
          py::arg("x"), py::arg("out") = py::none());
    m.def("reshape_and_cache", &reshape_and_cache, "write new tokens' K/V rows into the paged caches");
    m.def("plain_prefill", &plain_prefill, "flash_attention / flash_attention_gqa on plain arguments, else None");
    m.def("plain_varlen", &plain_varlen, "flash_attention_varlen on plain arguments, else None");
    m.def("plain_decode", &plain_decode, "paged_decode on plain arguments, else None");
    m.def("plain_write", &plain_write, "reshape_and_cache on plain arguments, else False");
    m.def("flash_gqa", &flash_gqa, "dense prefill with grouped-query attention");
    m.def("flash_varlen", &flash_varlen, "prefill over packed variable-length sequences");
}
