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
// The loads are non-temporal, and large writes store whole 128-byte lines
// (head_dim 64 and 128) through the L2 at device scope: cached loads of rows
// that the Infinity Cache no longer holds push the dirty lines of earlier
// kernels out of it, non-temporal stores wait for HBM, and stores left in the L2
// keep the next rows' loads waiting.  Measured on MI355X, us a call, Hkv=8, D=128, rows
// sliced from a fused projection, back to back / after 512 MiB were written /
// read / after the projection's rows were written: one token per workgroup with
// stores left in the L2 -> this
//    4096 tokens  6.3 / 10.2 / 10.3 /  9.0 ->  4.7 /  9.8 / 10.7 /  8.6
//    8192        13.8 / 17.6 / 17.3 / 14.0 -> 11.6 / 16.7 / 15.4 / 14.1
//   16384        23.6 / 29.6 / 26.4 / 23.9 -> 19.4 / 28.9 / 24.7 / 24.1
//   16384, Hkv=32  79 / 103 / 82 / 88      ->   77 / 101 / 80 / 87
// At 8192 tokens cached loads with non-temporal stores take 9.4 / 23.1 / 16.8 /
// 13.5 (16384, Hkv=32: 86 / 154 / 106 / 113), non-temporal both 11.9 / 16.6 /
// 16.0 / 16.8.
#include <hip/hip_runtime.h>

#include "attn_kernels.hpp"

namespace ak {

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

constexpr int kMaxWriteThreads = 256, kWave = 64;

// A store at device scope: written through the XCD's L2 (sc1).
__device__ __forceinline__ void store_through(u32x4 x, u32x4* p) {
    __builtin_amdgcn_global_store_b128((__attribute__((address_space(1))) u32x4*)p, x, "agent");
}

// One workgroup per (TOKENS tokens, group of up to 256 chunks): the token
// indices, their slots and the page arithmetic are wave-uniform (scalar
// registers); each lane moves one 16-byte chunk of K and one of V of each
// token, all loads issued before the first store.
template <int CPR, bool POW2_BS, int TOKENS>  // CPR = head_dim / 8 (0: runtime value)
__global__ void __launch_bounds__(kMaxWriteThreads)
cache_write_kernel(const u32x4* __restrict__ key, const u32x4* __restrict__ value, u32x4* __restrict__ k_cache,
                   u32x4* __restrict__ v_cache, const int64_t* __restrict__ slots, int num_tokens, int hkv, int cpr_rt,
                   int64_t key_stride, int64_t value_stride, int64_t num_slots, int bs, int bs_shift) {
    const int cpr = CPR ? CPR : cpr_rt;
    const int r = (int)(blockIdx.y * blockDim.x + threadIdx.x);  // = h * cpr + c: heads are contiguous
    if (r >= hkv * cpr) return;
    const int h = r / cpr, c = r - h * cpr;
    const int64_t t0 = (int64_t)blockIdx.x * TOKENS;
    int64_t slot[TOKENS];
    u32x4 kx[TOKENS], vx[TOKENS];
#pragma unroll
    for (int u = 0; u < TOKENS; ++u) {
        slot[u] = t0 + u < num_tokens ? slots[t0 + u] : -1;
        if (slot[u] >= num_slots) slot[u] = -1;
    }
#pragma unroll
    for (int u = 0; u < TOKENS; ++u)
        if (slot[u] >= 0) {
            kx[u] = __builtin_nontemporal_load(key + (t0 + u) * key_stride + r);
            vx[u] = __builtin_nontemporal_load(value + (t0 + u) * value_stride + r);
        }
#pragma unroll
    for (int u = 0; u < TOKENS; ++u)
        if (slot[u] >= 0) {
            const int64_t page = POW2_BS ? slot[u] >> bs_shift : slot[u] / bs;
            const int64_t dst = ((page * hkv + h) * bs + (slot[u] - page * bs)) * cpr + c;
            if (CPR % 8 == 0 && CPR > 0 && TOKENS > 1) {
                store_through(kx[u], k_cache + dst);
                store_through(vx[u], v_cache + dst);
            } else {
                k_cache[dst] = kx[u];
                v_cache[dst] = vx[u];
            }
        }
}

template <int CPR, int TOKENS>
static void launch_cw(const CacheWriteArgs& a, int per_token) {
    const int threads = per_token >= kMaxWriteThreads ? kMaxWriteThreads : (per_token + 63) / 64 * 64;
    const dim3 grid((unsigned)((a.num_tokens + TOKENS - 1) / TOKENS), (unsigned)((per_token + threads - 1) / threads));
    auto launch = [&](auto* kernel, int shift) {
        hipLaunchKernelGGL(kernel, grid, dim3(threads), 0, (hipStream_t)a.stream, static_cast<const u32x4*>(a.key),
                           static_cast<const u32x4*>(a.value), static_cast<u32x4*>(a.k_cache),
                           static_cast<u32x4*>(a.v_cache), a.slots, (int)a.num_tokens, (int)a.hkv,
                           (int)(a.head_dim / 8), a.key_stride / 8, a.value_stride / 8, a.num_blocks * a.bs, (int)a.bs,
                           shift);
    };
    if ((a.bs & (a.bs - 1)) == 0)
        launch(cache_write_kernel<CPR, true, TOKENS>, __builtin_ctzll((unsigned long long)a.bs));
    else
        launch(cache_write_kernel<CPR, false, TOKENS>, 0);
}

hipError_t cache_write_launch(const CacheWriteArgs& a) {
    const int per_token = (int)(a.hkv * (a.head_dim / 8));
    if (a.num_tokens == 0 || per_token == 0) return hipSuccess;
    // Two tokens per workgroup (four 16-byte loads in flight per lane) and stores
    // through the L2 from 8192 waves of chunks on: below that the misses of a
    // cold call overlap less, and its stores are done sooner in the L2 (2048
    // tokens, Hkv=8, D=128, after 512 MiB were written: 7.2 one token and L2,
    // 7.7 one and through, 8.2 two and through; back to back all 3.5).
    // Rows of part lines always stay in the L2 (8192 tokens, Hkv=5, D=40: 4.6
    // against 5.8 with non-temporal stores); two tokens help them where a token
    // leaves lanes of its wave idle (the same: 6.2 -> 3.8, cold 9.3 -> 8.9; not
    // D=96, Hkv=8: cold 14.2 -> 14.8), and past the 2^26 one-wave workgroups that
    // one launch holds.
    const bool whole_lines = a.head_dim == 128 || a.head_dim == 64;
    const bool two = whole_lines ? a.num_tokens * per_token >= 8192 * kWave
                                 : (per_token < kWave && a.num_tokens >= 8192) || a.num_tokens >= int64_t(1) << 25;
    if (a.head_dim == 128) two ? launch_cw<16, 2>(a, per_token) : launch_cw<16, 1>(a, per_token);
    else if (a.head_dim == 64) two ? launch_cw<8, 2>(a, per_token) : launch_cw<8, 1>(a, per_token);
    else two ? launch_cw<0, 2>(a, per_token) : launch_cw<0, 1>(a, per_token);
    return hipGetLastError();
}

}  // namespace ak
