// Paged KV-cache writer ("reshape and cache"): the step after a decode or a
// prefill that appends the new tokens' keys and values to the paged cache the
// decode kernel reads.  Not in the reference; its cache layout is the
// reference's (k/v cache [num_blocks, num_kv_heads, block_size, head_dim],
// attnkernels/reference.py:21-44, read at paged_decode.cu:95-96).
//
// Token t goes to page slot / block_size, row slot % block_size, for
// slot = slot_mapping[t]; a negative slot (padding) or one past the pool is
// skipped.  The move is a bit copy of 16-byte chunks, so fp16 and bf16 share
// the kernel.  Bound by memory: each chunk is read once and written once; one
// lane per chunk, consecutive lanes on consecutive chunks of one token, so a
// token's Hkv * head_dim elements move in whole 64-byte lines.
//
// The loads are cached (the projection that made the rows has usually just
// left them in the L2 or the Infinity Cache) and the stores of whole 128-byte
// lines (head_dim 64 and 128) are not: nothing reads them back soon, and they
// would push out the rows still to be read.  Two tokens per workgroup: four
// 16-byte loads in flight per lane.  Measured on MI355X, us a call, Hkv=8,
// D=128, rows sliced from a fused projection, one token per workgroup with
// non-temporal loads and cached stores -> this: 4096 tokens 8.0 -> 6.5, 8192
// 14.0 -> 10.9 (4.8 -> 6.1 TB/s), 16384 23.6 -> 21.5, 32768 53.3 -> 51.8.
// Only one of the two: 12.5 (cached loads), 13.1 (uncached stores) at 8192;
// three or four tokens 11.3.  Rows of part lines keep cached stores (8192
// tokens, Hkv=5, D=40: 4.6 against 5.8).
#include <hip/hip_runtime.h>

#include "attn_kernels.hpp"

namespace ak {

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

constexpr int kMaxWriteThreads = 256;

constexpr int kTokens = 2;  // per workgroup

// One workgroup per (kTokens tokens, group of up to 256 chunks): the token
// indices, their slots and the page arithmetic are wave-uniform (scalar
// registers); each lane moves one 16-byte chunk of K and one of V of each
// token, all loads issued before the first store.
template <int CPR, bool POW2_BS>  // CPR = head_dim / 8 (0: runtime value)
__global__ void __launch_bounds__(kMaxWriteThreads)
cache_write_kernel(const u32x4* __restrict__ key, const u32x4* __restrict__ value, u32x4* __restrict__ k_cache,
                   u32x4* __restrict__ v_cache, const int64_t* __restrict__ slots, int num_tokens, int hkv, int cpr_rt,
                   int64_t key_stride, int64_t value_stride, int64_t num_slots, int bs, int bs_shift) {
    const int cpr = CPR ? CPR : cpr_rt;
    const int r = (int)(blockIdx.y * blockDim.x + threadIdx.x);  // = h * cpr + c: heads are contiguous
    if (r >= hkv * cpr) return;
    const int h = r / cpr, c = r - h * cpr;
    const int64_t t0 = (int64_t)blockIdx.x * kTokens;
    int64_t slot[kTokens];
    u32x4 kx[kTokens], vx[kTokens];
#pragma unroll
    for (int u = 0; u < kTokens; ++u) {
        slot[u] = t0 + u < num_tokens ? slots[t0 + u] : -1;
        if (slot[u] >= num_slots) slot[u] = -1;
    }
#pragma unroll
    for (int u = 0; u < kTokens; ++u)
        if (slot[u] >= 0) {
            kx[u] = key[(t0 + u) * key_stride + r];
            vx[u] = value[(t0 + u) * value_stride + r];
        }
#pragma unroll
    for (int u = 0; u < kTokens; ++u)
        if (slot[u] >= 0) {
            const int64_t page = POW2_BS ? slot[u] >> bs_shift : slot[u] / bs;
            const int64_t dst = ((page * hkv + h) * bs + (slot[u] - page * bs)) * cpr + c;
            if (CPR % 8 == 0 && CPR > 0) {
                __builtin_nontemporal_store(kx[u], k_cache + dst);
                __builtin_nontemporal_store(vx[u], v_cache + dst);
            } else {
                k_cache[dst] = kx[u];
                v_cache[dst] = vx[u];
            }
        }
}

template <int CPR>
static void launch_cw(const CacheWriteArgs& a, dim3 grid, int threads, bool pow2, int shift) {
    const auto* k = static_cast<const u32x4*>(a.key);
    const auto* v = static_cast<const u32x4*>(a.value);
    auto* kc = static_cast<u32x4*>(a.k_cache);
    auto* vc = static_cast<u32x4*>(a.v_cache);
    const int cpr = (int)(a.head_dim / 8);
    auto launch = [&](auto* kernel) {
        hipLaunchKernelGGL(kernel, grid, dim3(threads), 0, (hipStream_t)a.stream, k, v, kc, vc, a.slots,
                           (int)a.num_tokens, (int)a.hkv, cpr, a.key_stride / 8, a.value_stride / 8,
                           a.num_blocks * a.bs, (int)a.bs, shift);
    };
    if (pow2) launch(cache_write_kernel<CPR, true>);
    else launch(cache_write_kernel<CPR, false>);
}

hipError_t cache_write_launch(const CacheWriteArgs& a) {
    const int per_token = (int)(a.hkv * (a.head_dim / 8));
    if (a.num_tokens == 0 || per_token == 0) return hipSuccess;
    const int threads = per_token >= kMaxWriteThreads ? kMaxWriteThreads : (per_token + 63) / 64 * 64;
    const dim3 grid((unsigned)((a.num_tokens + kTokens - 1) / kTokens), (unsigned)((per_token + threads - 1) / threads));
    const bool pow2 = (a.bs & (a.bs - 1)) == 0;
    const int shift = pow2 ? __builtin_ctzll((unsigned long long)a.bs) : 0;
    if (a.head_dim == 128)
        launch_cw<16>(a, grid, threads, pow2, shift);
    else if (a.head_dim == 64)
        launch_cw<8>(a, grid, threads, pow2, shift);
    else
        launch_cw<0>(a, grid, threads, pow2, shift);
    return hipGetLastError();
}

}  // namespace ak
