// The merge of the sparse attention's per-chunk (m, l, o) records, shared by
// the attention launch (attention.hip) and by the launch that runs it beside
// the next layer's selection count (select.hip).
#pragma once

#include <hip/hip_runtime.h>

#include <cmath>
#include <cstdint>

#include "hs_device.hpp"

namespace hs {

// Token ids per partial workgroup: the shortest of 32, 64 and 128 that makes at
// most 256 workgroups, one for each CU.  A workgroup is a chain of round trips
// (membership, rows, record), and 128 ids on a quarter of the CUs make each
// of its steps longer than it need be.  Eight pipelined layers of 2048 / 8192
// / 16384 tokens take 226 / 255 / 290 us against 275 / 297 / 321 with 128 ids
// everywhere, one layer (V rows only) of 3001 / 8192 / 16384 23.0 / 26.4 /
// 32.7 against 24.9 / 28.0 / 33.8.  More workgroups than CUs do not pay: 32 ids
// at 16384 tokens 35.2 us, 64 at 32768 45.1 against 43.8, twice the records.
// The softmax weights are rounded to F16 against their chunk's maximum, so a
// shorter chunk is also nearer 64 bits: 1.3e-4 with 32 ids, 1.5e-4 with 64,
// 1.65e-4 with 128.  What it costs is the merge: the V-only call alone with 2 %
// of the ids selected takes 9.7 us against 8.5 at 8192 tokens (9.9 / 9.1 at
// 16384), with 20 % 10.2 against 10.9.  (256 CUs are the whole GPU's; the
// workspace sizes follow the chunks, so they do not depend on the device.)
constexpr uint32_t kAttnChunk = 128;
constexpr uint32_t kAttnShort = 256 * 32, kAttnMiddle = 256 * 64;
inline uint32_t attn_chunk(uint32_t n) { return n <= kAttnShort ? 32u : n <= kAttnMiddle ? 64u : kAttnChunk; }
inline uint32_t attn_chunks(uint32_t n) { return (n + attn_chunk(n) - 1) / attn_chunk(n); }
constexpr uint32_t kAttnRecord = 2 + 128;  // m, l, o[128] per (chunk, query head)

// Merge the per-chunk (m, l, o) records of query head h, channels
// 32*channel_group .. +31, by one kCombineThreads workgroup.  Every record
// value a workgroup needs is requested up front, since none depends on
// another: the o values of this thread's channel over every 16th chunk, and
// one chunk's (m, l) per thread.
// Then the chunk weights exp(m_i - max m) and their l sum, 16 rows of 32
// threads each summing the weighted o of their chunks, and the 16 partial
// sums added in LDS.
constexpr uint32_t kMaxChunks = 65536 / kAttnChunk;
constexpr uint32_t kCombineThreads = 512;
constexpr uint32_t kCombineRows = 16;  // chunks r, r + 16, ... per row of 32 threads
static_assert(kMaxChunks <= kCombineThreads, "one chunk weight per thread");
struct CombineLds {
    float weight[kMaxChunks];
    float red[8];
    float acc16[kCombineRows][33];
};
// kFirst: o values per thread, at least ceil(chunks / kCombineRows).
template <uint32_t kFirst>
__device__ __forceinline__ void combine_batch(const float* __restrict__ part, uint32_t chunks,
                                              float* __restrict__ out, uint32_t h,
                                              uint32_t channel_group, CombineLds& lds) {
    auto& weight = lds.weight;
    auto& red = lds.red;
    auto& acc16 = lds.acc16;
    const uint32_t g = h >> 2, j = h & 3u, tid = threadIdx.x;
    const uint32_t lane = tid & 63u, wave = tid >> 6;
    const float* recs = part + static_cast<size_t>(g) * chunks * 4 * kAttnRecord + j * kAttnRecord;
    const uint32_t c = tid & 31u, r = tid >> 5, ch = channel_group * 32 + c;
    const uint32_t last = chunks - 1;  // reads past the last chunk are clamped to it
    float v[kFirst];
#pragma unroll
    for (uint32_t u = 0; u < kFirst; ++u)
        v[u] = recs[min(r + kCombineRows * u, last) * 4 * kAttnRecord + 2 + ch];
    const float* mine = recs + min(tid, last) * 4 * kAttnRecord;
    const float m_rec = mine[0], l_rec = mine[1];
    const float m = tid < chunks ? m_rec : -INFINITY;
    const float l = tid < chunks ? l_rec : 0.0f;
    float top = wave_max_f32(m);
    if (lane == 0) red[wave] = top;
    __syncthreads();
    top = red[0];
#pragma unroll
    for (uint32_t w = 1; w < 8; ++w) top = fmaxf(top, red[w]);
    const float w_self = (m == -INFINITY || top == -INFINITY) ? 0.0f : __expf(m - top);
    weight[tid] = w_self;
    __syncthreads();
    const float lsum = wave_sum_f32(l * w_self);
    __syncthreads();  // every wave has read red[] before it is reused
    if (lane == 0) red[wave] = lsum;
    __syncthreads();
    float L = 0.0f;
#pragma unroll
    for (uint32_t w = 0; w < 8; ++w) L += red[w];
    // the weights are read before any is used (a read inside the test
    // below would make each term wait for its own LDS round trip); a zero
    // weight still skips its term, whose o may be inf or NaN
    float wv[kFirst];
#pragma unroll
    for (uint32_t u = 0; u < kFirst; ++u) wv[u] = weight[r + kCombineRows * u];
    float a = 0.0f;
#pragma unroll
    for (uint32_t u = 0; u < kFirst; ++u) {
        const uint32_t i = r + kCombineRows * u;
        if (i < chunks && wv[u] != 0.0f) a = __builtin_fmaf(v[u], wv[u], a);
    }
    acc16[r][c] = a;
    __syncthreads();
    if (tid < 32) {
        float sum = 0.0f;
#pragma unroll
        for (uint32_t k = 0; k < kCombineRows; ++k) sum += acc16[k][tid];
        // no selected row: NaN, as a fully masked softmax row gives, never a
        // silent zero (the reference refuses an empty selection)
        out[h * 128 + ch] = L > 0.0f ? sum / L : __builtin_nanf("");
    }
}

// The batch is chosen by the number of chunks: 4, 16 or 32 values per thread
// for up to 64, 256 and 512 of them (the order of the sum does not depend on
// it).  A batch whose later values were read one by
// one in a loop made n = 65536 wait a round trip per 16 chunks: its layer
// takes 72.8 us with 32 values at once against 77.6.  The short batch takes
// 28.0 against 28.3 us at n = 1024 and 28.4 against 29.0 at 4096, where most
// of 16 values are the last chunk's again.
__device__ __forceinline__ void combine_records(const float* __restrict__ part, uint32_t chunks,
                                                float* __restrict__ out, uint32_t h,
                                                uint32_t channel_group, CombineLds& lds) {
    static_assert(kMaxChunks <= 32 * kCombineRows, "the widest batch covers every chunk");
    if (chunks <= 4 * kCombineRows)
        combine_batch<4>(part, chunks, out, h, channel_group, lds);
    else if (chunks <= 16 * kCombineRows)
        combine_batch<16>(part, chunks, out, h, channel_group, lds);
    else
        combine_batch<32>(part, chunks, out, h, channel_group, lds);
}

}  // namespace hs
