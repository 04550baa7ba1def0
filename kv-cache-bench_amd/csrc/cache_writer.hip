// The cache writers on the GPU: the contiguous cache [B][Hkv][max_len][D] into the paged pool
// [blocks][Hkv][page][D] through the block table, as the reference's host-side scatter_to_paged
// (src/reference.hpp:60-68) and quantize_to_paged_i8 (src/reference.cpp:32-51) do, with the same
// bytes and scales.
//
// A block's live rows are contiguous in both layouts, and a row is a whole number of 16-byte words (D
// is 64 or 128). Both kernels are bound by the card's mixed read and write rate. A call that moves
// kStreamBytes or more reads the contiguous cache with non-temporal loads: it is read once, and the
// pool's lines, which the next decode step reads, keep the caches to themselves. A smaller call finds
// the rows its prompt's projection has just written in the 256 MB memory-side cache, which ordinary
// loads use best. (MI355X, us of a prompt's K and then its V, ordinary / non-temporal, freshly written
// and then the same buffers again and again; 8 KV heads, head_dim 128, page 64: fp32, 64 sequences of up
// to 300 tokens, 79 MB a call, 25.3 / 27.2 and 25.5 / 32.2; fp16, 16 of up to 4096, 131 MB, 51.9 / 44.1
// and 45.0 / 51.1; 16 of 4096, 268 MB, 108.9 / 81.7 and 101.5 / 82.0. The line lies where the rows and
// pools of K and V together outgrow that cache. Non-temporal stores were slower.)
#include <algorithm>

#include "kvb_kernels.hpp"

namespace kvbk {
namespace {

constexpr int kWriterThreads = 256;
constexpr long long kStreamBytes = 128ll << 20;  // read and written

typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));

// 16 bytes of the contiguous cache, STREAM: with the non-temporal policy.
template <bool STREAM>
__device__ __forceinline__ u32x4_t load_word(const u32x4_t* p) {
    if constexpr (STREAM) return __builtin_nontemporal_load(p);
    else return *p;
}

// A workgroup copies kWriterThreads * U 16-byte words of consecutive tokens (U 2, 8 KB: 32 fp16 rows at
// head_dim 128) of one (KV head, sequence), whatever the page size: the loads do not wait for the block
// ids, which each lane looks up for its own rows while they are in flight. (1, 2 and 4 words per thread: 2
// is the fastest or within 4% of it from 0.2 MB to 1 GB; of the calls that stream, 4 by 1-2%.)
constexpr int scatter_words(bool stream) { return stream ? 4 : 2; }
template <bool STREAM>
__global__ __launch_bounds__(kWriterThreads) void scatter_kernel(CacheWriteParams p) {
    constexpr int U = scatter_words(STREAM);
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
            x[u] = load_word<STREAM>(src + min(u * kWriterThreads + (int)threadIdx.x, n - 1));
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

// Groups of 4 values a thread may hold: a workgroup holds a block of up to 64 KB (page 128 at head_dim 128).
constexpr int kQuantRegs = 16;

// The live rows of one (KV head, sequence, logical block) as groups of 4 values.
struct QuantBlock {
    const u32x4_t* src;
    long long n4;
    template <bool STREAM>
    __device__ float4 at(long long w) const { return __builtin_bit_cast(float4, load_word<STREAM>(src + w)); }
};
__device__ __forceinline__ QuantBlock quant_block(const CacheWriteParams& p, int kvh, int b, int blk_i) {
    const int t0 = blk_i * p.page_size;
    const int rows = max(0, min(live_len(p.seq_lens, b, p.len_cap) - t0, p.page_size));
    return {reinterpret_cast<const u32x4_t*>(static_cast<const float*>(p.contig) +
                                             (((size_t)b * p.num_kv_heads + kvh) * p.max_len + t0) * p.head_dim),
            (long long)rows * p.head_dim / 4};
}

// The values of a block held in registers between its max and its quantisation: up to T * R groups.
template <int T, int R, bool STREAM>
__device__ __forceinline__ void quantize_held(const CacheWriteParams& p, const QuantBlock& q, size_t slot, int tid) {
    float4 v[R];
    float amax = 0.0f;
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const int w = tid + r * T;
        v[r] = w < q.n4 ? q.at<STREAM>(w) : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    }
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

__device__ __forceinline__ size_t quant_slot(const CacheWriteParams& p, int kvh, int b, int blk_i) {
    return (size_t)p.block_table[(size_t)b * p.max_blocks + blk_i] * p.num_kv_heads + kvh;
}

// T = 64: a wave per block, four blocks per workgroup, without a barrier. T = 256: the workgroup.
template <int T, int R, bool STREAM>
__global__ __launch_bounds__(kWriterThreads) void quantize_kernel(CacheWriteParams p) {
    const int kvh = blockIdx.x, b = blockIdx.y;
    const int blk_i = blockIdx.z * (kWriterThreads / T) + threadIdx.x / T;
    // (blk_i may lie up to three blocks past max_len: no live rows)
    const QuantBlock q = quant_block(p, kvh, b, blk_i);
    if (q.n4 == 0) return;  // uniform over the team, before the barrier of a workgroup's team
    quantize_held<T, R, STREAM>(p, q, quant_slot(p, kvh, b, blk_i), threadIdx.x % T);
}

// Pages whose blocks may not fit in registers: a block is read twice by the workgroup, the second time
// from L2 where it holds it. HELD: one that does fit is held, for batches whose sequences all end before
// such a page fills (one of 100 tokens, 8 KV heads, page 256: 5.2 us against 7.2). Where blocks do not fit,
// the held form's registers cost workgroups per CU (8 ragged up to 4096, page 129: 34.4 us against 30.0).
template <bool HELD>
__global__ __launch_bounds__(kWriterThreads) void quantize_large_kernel(CacheWriteParams p) {
    const int kvh = blockIdx.x, b = blockIdx.y, blk_i = blockIdx.z;
    const QuantBlock q = quant_block(p, kvh, b, blk_i);
    if (q.n4 == 0) return;  // uniform over the workgroup, before the barrier in team_max
    const size_t slot = quant_slot(p, kvh, b, blk_i);
    if (HELD && q.n4 <= kWriterThreads * kQuantRegs) {  // uniform
        quantize_held<kWriterThreads, kQuantRegs, false>(p, q, slot, threadIdx.x);
        return;
    }
    uint32_t* dst = reinterpret_cast<uint32_t*>(static_cast<int8_t*>(p.paged) + slot * p.page_size * p.head_dim);
    float amax = 0.0f;
    for (long long w = threadIdx.x; w < q.n4; w += kWriterThreads) amax = abs_max4(amax, q.at<false>(w));
    const float scale = team_max<kWriterThreads>(amax) / 127.0f;
    if (threadIdx.x == 0) p.scales[slot] = scale;
    for (long long w = threadIdx.x; w < q.n4; w += kWriterThreads) dst[w] = quantize4(q.at<false>(w), scale);
}

// The quantiser's forms: by the groups of 4 values a block can hold (max_len bounds them too), and for
// blocks of up to 8 KB by how many there are. A wave per block keeps a block's divisions to one wave:
// the faster where every SIMD has a wave (8 x 8192 tokens at page 16: 56.8 us, against 61.6 with the
// workgroup on one block), the slower where the chip is idle (100 tokens, 8 KV heads, page 16, cold: 6.8
// against 5.0). The line lies at a wave per SIMD: between 0.6 and 1.1 blocks per SIMD the two cross.
template <bool STREAM>
void launch_quantize(const CacheWriteParams& p, int batch, int max_blocks_used, hipStream_t s, const Marks& m) {
    const dim3 block(kWriterThreads);
    const long long n4 = std::min(p.page_size, p.max_len) * (p.head_dim / 4ll);
    const bool waves = n4 <= 64 * 8 && p.live_blocks >= 4ll * p.cus;
    const int teams = waves ? kWriterThreads / 64 : 1;
    const dim3 grid(p.num_kv_heads, batch, (max_blocks_used + teams - 1) / teams);
    if (waves) launch_marked(quantize_kernel<64, 8, STREAM>, grid, block, s, m, p);
    else if (n4 <= kWriterThreads * 2) launch_marked(quantize_kernel<kWriterThreads, 2, STREAM>, grid, block, s, m, p);
    else if (n4 <= kWriterThreads * 8) launch_marked(quantize_kernel<kWriterThreads, 8, STREAM>, grid, block, s, m, p);
    else if (n4 <= kWriterThreads * kQuantRegs) launch_marked(quantize_kernel<kWriterThreads, kQuantRegs, STREAM>, grid, block, s, m, p);
    else if (std::min(p.page_size, p.longest) * (p.head_dim / 4ll) <= kWriterThreads * kQuantRegs)
        launch_marked(quantize_large_kernel<true>, grid, block, s, m, p);
    else launch_marked(quantize_large_kernel<false>, grid, block, s, m, p);
}

}  // namespace

hipError_t launch_write_paged(const CacheWriteParams& p, int batch, int max_blocks_used, hipStream_t s,
                              const Marks& m) {
    const long long values = p.live_tokens * p.num_kv_heads * p.head_dim;
    const bool stream = values * (p.quantize ? 5 : 2 * p.elem_size) >= kStreamBytes;
    if (p.quantize) {
        if (stream) launch_quantize<true>(p, batch, max_blocks_used, s, m);
        else launch_quantize<false>(p, batch, max_blocks_used, s, m);
        return hipGetLastError();
    }
    const int tokens = (kWriterThreads * scatter_words(stream)) >> p.row_shift;
    const long long runs = (p.max_len + (long long)tokens - 1) / tokens;
    const dim3 grid(p.num_kv_heads, batch, (unsigned)(runs < 65535 ? runs : 65535)), block(kWriterThreads);
    if (stream) launch_marked(scatter_kernel<true>, grid, block, s, m, p);
    else launch_marked(scatter_kernel<false>, grid, block, s, m, p);
    return hipGetLastError();
}

}  // namespace kvbk
