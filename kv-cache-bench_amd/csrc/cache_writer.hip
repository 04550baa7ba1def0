// The cache writers on the GPU: the contiguous cache [B][Hkv][max_len][D] into the paged pool
// [blocks][Hkv][page][D] through the block table, as the reference's host-side scatter_to_paged
// (src/reference.hpp:60-68) and quantize_to_paged_i8 (src/reference.cpp:32-51) do, with the same
// bytes and scales.
//
// A block's live rows are contiguous in both layouts, and a row is a whole number of 16-byte words (D
// is 64 or 128). Both kernels are bound by the card's mixed read and write rate, and both read the
// contiguous cache with non-temporal loads: it is read once, and the pool's lines, which the next decode
// step reads, keep the caches to themselves. (MI355X: 16 ragged sequences up to 4096 tokens, 8 KV heads,
// fp16, page 16, 139 MB read and written: 29.9 us with ordinary loads, 24.5 with non-temporal ones;
// non-temporal stores as well: 28.1. 8 x 8192 tokens quantised to int8, page 64, 336 MB: 69.6, 59.1 and
// 62.1.)
#include "kvb_kernels.hpp"

namespace kvbk {
namespace {

constexpr int kWriterThreads = 256;
constexpr int kScatterWords = 4;

typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));

// A workgroup copies kWriterThreads * kScatterWords 16-byte words of consecutive tokens (16 KB: 64
// fp16 rows at head_dim 128) of one (KV head, sequence), whatever the page size: the loads do not wait
// for the block ids, which each lane looks up for its own rows while they are in flight. (One
// workgroup per block, with one word in flight per thread at 16-token pages, took 33.7 us where this
// takes 24.5; 1, 2, 4, 8 and 16 words per thread are within 3% of each other.)
__global__ __launch_bounds__(kWriterThreads) void scatter_kernel(CacheWriteParams p) {
    constexpr int U = kScatterWords;
    const int kvh = blockIdx.x, b = blockIdx.y;
    const int len = live_len(p.seq_lens, b, p.len_cap);
    const int shift = p.row_shift, tokens = (kWriterThreads * U) >> shift;
    // (one turn, but for sequences of more runs than a grid has)
    for (long long t00 = (long long)blockIdx.z * tokens; t00 < len; t00 += (long long)gridDim.z * tokens) {
        const int t0 = (int)t00, n = min(len - t0, tokens) << shift;  // live words
        const u32x4_t* src = static_cast<const u32x4_t*>(p.contig) +
                             ((((size_t)b * p.num_kv_heads + kvh) * p.max_len + t0) << shift);
        u32x4_t x[U];
    #pragma unroll
        for (int u = 0; u < U; ++u)  // (past the end: the last live word again, not written)
            x[u] = __builtin_nontemporal_load(src + min(u * kWriterThreads + (int)threadIdx.x, n - 1));
        size_t dst[U];
    #pragma unroll
        for (int u = 0; u < U; ++u) {
            const int w = min(u * kWriterThreads + (int)threadIdx.x, n - 1);
            const int t = t0 + (w >> shift), bi = fast_div(t, p.page_div);
            const size_t blk = (size_t)p.block_table[(size_t)b * p.max_blocks + bi];
            const size_t row = (blk * p.num_kv_heads + kvh) * p.page_size + (t - bi * p.page_size);
            dst[u] = (row << shift) + (w & ((1 << shift) - 1));
        }
    #pragma unroll
        for (int u = 0; u < U; ++u)
            if (u * kWriterThreads + (int)threadIdx.x < n) static_cast<u32x4_t*>(p.paged)[dst[u]] = x[u];
    }
}

// The max of x over a team of T threads: a wave, or the whole workgroup.
template <int T>
__device__ __forceinline__ float team_max(float x) {
    for (int o = 32; o > 0; o >>= 1) x = fmaxf(x, __shfl_xor(x, o));
    if constexpr (T == 64) {
        return x;
    } else {
        __shared__ float s_max[kWriterThreads / 64];
        if ((threadIdx.x & 63) == 0) s_max[threadIdx.x >> 6] = x;
        __syncthreads();
        float m = s_max[0];
        for (int w = 1; w < kWriterThreads / 64; ++w) m = fmaxf(m, s_max[w]);
        return m;
    }
}

// x / scale rounded half to even and clamped to +-127 (scale > 0), as the reference's
// int8(clamp(nearbyint(x / scale), -127, 127)); the division is IEEE (correctly rounded).
__device__ __forceinline__ uint32_t quantize_byte(float x, float scale) {
    const float q = fminf(fmaxf(__builtin_rintf(x / scale), -127.0f), 127.0f);
    return (uint32_t)(uint8_t)(int8_t)(int)q;
}

__device__ __forceinline__ float abs_max4(float m, const float4& v) {
    return fmaxf(fmaxf(m, fmaxf(fabsf(v.x), fabsf(v.y))), fmaxf(fabsf(v.z), fabsf(v.w)));
}

__device__ __forceinline__ uint32_t quantize4(const float4& v, float scale) {
    if (!(scale > 0.0f)) return 0u;  // an all-zero slice: every byte 0
    return quantize_byte(v.x, scale) | quantize_byte(v.y, scale) << 8 | quantize_byte(v.z, scale) << 16 |
           quantize_byte(v.w, scale) << 24;
}

// The live rows of one (KV head, sequence, logical block) as groups of 4 values.
struct QuantBlock {
    const u32x4_t* src;
    long long n4;
    __device__ float4 at(int w) const { return __builtin_bit_cast(float4, __builtin_nontemporal_load(src + w)); }
};
__device__ __forceinline__ QuantBlock quant_block(const CacheWriteParams& p, int kvh, int b, int blk_i) {
    const int t0 = blk_i * p.page_size;
    const int rows = max(0, min(live_len(p.seq_lens, b, p.len_cap) - t0, p.page_size));
    return {reinterpret_cast<const u32x4_t*>(static_cast<const float*>(p.contig) +
                                             (((size_t)b * p.num_kv_heads + kvh) * p.max_len + t0) * p.head_dim),
            (long long)rows * p.head_dim / 4};
}

// A block of up to T * R groups is read once and kept in registers between its max and its
// quantisation. T = 64: a wave per block, four blocks per workgroup, without a barrier (blocks of up to
// 8 KB: 16 tokens at head_dim 128; 8 x 8192 tokens at page 16: 56.8 us, against 61.6 with the whole
// workgroup on one block). T = 256: the workgroup.
template <int T, int R>
__global__ __launch_bounds__(kWriterThreads) void quantize_kernel(CacheWriteParams p) {
    const int kvh = blockIdx.x, b = blockIdx.y, tid = threadIdx.x % T;
    const int blk_i = blockIdx.z * (kWriterThreads / T) + threadIdx.x / T;
    // (blk_i may lie up to three blocks past max_len: no live rows)
    const QuantBlock q = quant_block(p, kvh, b, blk_i);
    if (q.n4 == 0) return;  // uniform over the team, before the barrier of a workgroup's team
    float4 v[R];
    float amax = 0.0f;
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const int w = tid + r * T;
        v[r] = w < q.n4 ? q.at(w) : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    }
    const size_t slot = (size_t)p.block_table[(size_t)b * p.max_blocks + blk_i] * p.num_kv_heads + kvh;
#pragma unroll
    for (int r = 0; r < R; ++r) amax = abs_max4(amax, v[r]);
    const float scale = team_max<T>(amax) / 127.0f;
    if (tid == 0) p.scales[slot] = scale;
    uint32_t* dst = reinterpret_cast<uint32_t*>(static_cast<int8_t*>(p.paged) + slot * p.page_size * p.head_dim);
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const int w = tid + r * T;
        if (w < q.n4) dst[w] = quantize4(v[r], scale);
    }
}

// Larger blocks are read twice by the workgroup, the second time from L2 where it holds them.
__global__ __launch_bounds__(kWriterThreads) void quantize_large_kernel(CacheWriteParams p) {
    const int kvh = blockIdx.x, b = blockIdx.y, blk_i = blockIdx.z;
    const QuantBlock q = quant_block(p, kvh, b, blk_i);
    if (q.n4 == 0) return;  // uniform over the workgroup, before the barrier in team_max
    const float4* src = reinterpret_cast<const float4*>(q.src);
    const size_t slot = (size_t)p.block_table[(size_t)b * p.max_blocks + blk_i] * p.num_kv_heads + kvh;
    uint32_t* dst = reinterpret_cast<uint32_t*>(static_cast<int8_t*>(p.paged) + slot * p.page_size * p.head_dim);
    float amax = 0.0f;
    for (long long w = threadIdx.x; w < q.n4; w += kWriterThreads) amax = abs_max4(amax, src[w]);
    const float scale = team_max<kWriterThreads>(amax) / 127.0f;
    if (threadIdx.x == 0) p.scales[slot] = scale;
    for (long long w = threadIdx.x; w < q.n4; w += kWriterThreads) dst[w] = quantize4(src[w], scale);
}

}  // namespace

hipError_t launch_write_paged(const CacheWriteParams& p, int batch, int max_blocks_used, hipStream_t s,
                              const Marks& m) {
    const dim3 block(kWriterThreads);
    if (!p.quantize) {
        const int tokens = (kWriterThreads * kScatterWords) >> p.row_shift;
        const long long runs = (p.max_len + (long long)tokens - 1) / tokens;
        launch_marked(scatter_kernel, dim3(p.num_kv_heads, batch, (unsigned)(runs < 65535 ? runs : 65535)), block, s, m, p);
        return hipGetLastError();
    }
    const long long n4 = (long long)p.page_size * p.head_dim / 4;
    const int teams = n4 <= 64 * 8 ? kWriterThreads / 64 : 1;
    const dim3 grid(p.num_kv_heads, batch, (max_blocks_used + teams - 1) / teams);
    if (n4 <= 64 * 8) launch_marked(quantize_kernel<64, 8>, grid, block, s, m, p);
    else if (n4 <= kWriterThreads * 8) launch_marked(quantize_kernel<kWriterThreads, 8>, grid, block, s, m, p);
    else if (n4 <= kWriterThreads * 16) launch_marked(quantize_kernel<kWriterThreads, 16>, grid, block, s, m, p);
    else launch_marked(quantize_large_kernel, grid, block, s, m, p);
    return hipGetLastError();
}

}  // namespace kvbk
