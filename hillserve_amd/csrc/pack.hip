// Kernel #3 — physical union, packed-workspace build and row-map gather.
//
//  * hs_gqa_physical_union: runtime/gqa_pack.hpp:12-22.  One bitmap over the
//    visible ids per query head, duplicate and future ids rejected, then an
//    order-preserving compaction of their OR -> sorted unique ids.
//  * hs_gqa_pack: runtime/gqa_pack.hpp:26-58, byte for byte: K
//    [slot][Qhead][128], V transposed [Qhead][128][slot], mask
//    [Qhead][qpad][slot] = 0 where id <= position[q], -inf elsewhere, zero
//    K/V padding.  Rows come from the device hot pool (row r's K[8][128] at
//    k_pool + r * row_bytes, its V[8][128] at v_pool + r * row_bytes; the
//    reference's 4096 B records are k_pool = pool, v_pool = pool + 2048)
//    through an optional id -> row map.
//  * hs_gqa_gather_rows: runtime/gqa_prefetch_cuda.cu:12-22 (row map
//    >=0 prefetched, <=-2 miss row, -1 zero).
// K and V for a (head, 64-slot) block are staged in LDS so both the K rows
// and the transposed V rows leave as contiguous runs.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>

#include "hs_device.hpp"
#include "hs_internal.hpp"

namespace hs {
namespace {

constexpr uint32_t kMaxVisible = 66048;  // gqa_pack.hpp:14,29

__global__ void fill_u32_kernel(uint32_t* __restrict__ dst, uint32_t count, uint32_t value) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < count) dst[i] = value;
}

}  // namespace

void launch_fill_u32(uint32_t* dst, uint32_t count, uint32_t value, hipStream_t stream) {
    hipLaunchKernelGGL(fill_u32_kernel, dim3((count + 255) / 256), dim3(256), 0, stream, dst, count,
                       value);
}

namespace {

// Physical union in two launches.  A head's list becomes a bitmap over the
// visible ids in one workgroup's LDS (at most 66048 ids: 8.3 KB), where the
// atomic's old word shows a duplicate, and is written out whole, so nothing
// needs clearing first; the second launch ORs the 32 bitmaps and compacts.
// Latency-bound: 32 x 6553 ids (0.8 MB in, 0.3 MB of bitmaps) take two
// dependent launches of a few memory round trips each.  The five launches
// before it (two fills, atomics on one global word per id, count, write)
// took 13.4 us more at 32768 visible ids (union and pack 73.1 -> 59.7 us),
// 6.1 us more at 8192 (23.8 -> 17.7 us) and 13.9 us more at 48001 (score,
// cover and union 97.1 -> 83.2 us).
constexpr uint32_t kUnionThreads = 1024;
constexpr uint32_t kMaxUnionWords = (kMaxVisible + 31) / 32;  // 2064
constexpr uint32_t kUnionBatch = 8;  // ids per thread requested before any is used

// One workgroup per head: bitmap of its ids, and whether it holds a
// duplicate or future id.
__global__ void __launch_bounds__(kUnionThreads)
union_mark_kernel(const uint32_t* __restrict__ ids, const uint32_t* __restrict__ lens,
                  uint32_t ids_stride, uint32_t visible, uint32_t* __restrict__ bitmaps,
                  uint32_t* __restrict__ bad_heads) {
    __shared__ uint32_t bits[kMaxUnionWords];
    __shared__ uint32_t bad;
    const uint32_t h = blockIdx.x, tid = threadIdx.x, words = (visible + 31) / 32;
    const uint32_t len = lens[h];
    const uint32_t* list = ids + static_cast<size_t>(h) * ids_stride;
    for (uint32_t w = tid; w < words; w += kUnionThreads) bits[w] = 0;
    if (tid == 0) bad = 0;
    __syncthreads();
    bool mine_bad = false;
    for (uint64_t first = 0; first < len; first += kUnionThreads * kUnionBatch) {
        uint32_t id[kUnionBatch];
#pragma unroll
        for (uint32_t u = 0; u < kUnionBatch; ++u) {  // (len >= 1 here: the index is clamped)
            const uint64_t j = first + u * kUnionThreads + tid;
            id[u] = list[j < len ? j : len - 1u];
        }
#pragma unroll
        for (uint32_t u = 0; u < kUnionBatch; ++u) {
            if (first + u * kUnionThreads + tid >= len) continue;
            if (id[u] >= visible) {
                mine_bad = true;
                continue;
            }
            const uint32_t bit = 1u << (id[u] & 31u);
            mine_bad |= (atomicOr(&bits[id[u] >> 5], bit) & bit) != 0;
        }
    }
    if (mine_bad) bad = 1;
    __syncthreads();
    for (uint32_t w = tid; w < words; w += kUnionThreads)
        bitmaps[static_cast<size_t>(h) * words + w] = bits[w];
    if (tid == 0) bad_heads[h] = bad;
}

// Workgroup b writes the union's ids of bitmap words 64 b .. 64 b + 63.  Its
// place in the output is the number of union ids in the words before them,
// which it counts itself from the bitmaps (at most 264 KB from L2), so the
// workgroups wait for nothing.
constexpr uint32_t kUnionWords = 64;
__global__ void __launch_bounds__(kUnionThreads)
union_write_kernel(const uint32_t* __restrict__ bitmaps, const uint32_t* __restrict__ bad_heads,
                   uint32_t visible, uint32_t* __restrict__ out, uint32_t* __restrict__ out_n,
                   hs_status_t* __restrict__ status) {
    __shared__ uint32_t own[kUnionWords], first_at[kUnionWords];
    __shared__ uint32_t before[kUnionThreads / 64];
    const uint32_t tid = threadIdx.x, lane = tid & 63u, words = (visible + 31) / 32;
    const uint32_t first = blockIdx.x * kUnionWords;
    const uint32_t end = first + kUnionWords < words ? first + kUnionWords : words;
    if (tid < kUnionWords) own[tid] = 0;
    __syncthreads();
    uint32_t count = 0;
    for (uint32_t w = tid; w < end; w += kUnionThreads) {
        uint32_t v[32], any = 0;
#pragma unroll
        for (uint32_t h = 0; h < 32; ++h) v[h] = bitmaps[static_cast<size_t>(h) * words + w];
#pragma unroll
        for (uint32_t h = 0; h < 32; ++h) any |= v[h];
        if (w < first) count += static_cast<uint32_t>(__popc(any));
        else own[w - first] = any;
    }
    count = wave_sum_u32(count);
    if (lane == 0) before[tid >> 6] = count;
    __syncthreads();
    if (tid < kUnionWords) {  // wave 0
        uint32_t at = 0;
#pragma unroll
        for (uint32_t w = 0; w < kUnionThreads / 64; ++w) at += before[w];
        const uint32_t c = static_cast<uint32_t>(__popc(own[tid]));
        const uint32_t x = wave_inclusive_sum_u32(c);
        first_at[tid] = at + x - c;
        if (blockIdx.x == gridDim.x - 1 && tid == kUnionWords - 1) *out_n = at + x;
        if (blockIdx.x == 0) {
            const uint64_t any_bad = __ballot(tid < 32 && bad_heads[tid & 31u] != 0);
            if (tid == 0) {
                hs_status_t st{};
                st.code = any_bad ? HS_ERR_DUPLICATE : HS_OK;
                *status = st;
            }
        }
    }
    __syncthreads();
    for (uint32_t i = tid; i < kUnionWords * 32; i += kUnionThreads) {
        const uint32_t w = i >> 5, b = i & 31u, x = own[w];
        if ((x >> b) & 1u)
            out[first_at[w] + static_cast<uint32_t>(__popc(x & ((1u << b) - 1u)))] = first * 32 + i;
    }
}

// Source of one (slot, head) pair of the packed layout.
struct PoolSource {
    const uint8_t* pool;   // K rows
    uint32_t pool_rows;
    uint32_t row_bytes;
    int64_t v_delta;       // a row's V segment sits v_delta bytes from its K segment
    const int32_t* row_of_id;
    uint32_t max_id;
    const uint32_t* ids;
    const uint32_t* lens;
    uint32_t ids_stride;
};

struct MapSource {
    const uint16_t* prefetched;
    const uint16_t* misses;
    const int32_t* map;
    uint32_t prefetched_rows, miss_rows;
};

// A row every slot may read when it has none of its own (its bytes are
// discarded): the pool's first row, or the first prefetched or miss record;
// null when there is no source at all.  For the pool, row 0's K and V
// segments exist whenever pool_rows > 0.
__device__ __forceinline__ const uint8_t* fallback_row(const PoolSource& ps, const MapSource& ms,
                                                       bool pack) {
    if (pack) return ps.pool_rows > 0 ? ps.pool : nullptr;
    if (ms.prefetched && ms.prefetched_rows > 0) return reinterpret_cast<const uint8_t*>(ms.prefetched);
    if (ms.misses && ms.miss_rows > 0) return reinterpret_cast<const uint8_t*>(ms.misses);
    return nullptr;
}

// Grid (ceil(count/kSlots), 32 heads), 4 threads per slot.  kPack selects the
// source.  64 slots at a time; 32 up to kShortSlots, where 64 would leave the
// chip's 8 workgroups per CU unfilled (one workspace: gather of 1664 slots 9.6
// -> 8.3 us, of 3296 18.1 -> 17.1, pack of 3296 22.5 -> 21.7) and above which
// the shorter runs of V cost more than the finer split gives (6560 slots:
// gather 43.5 -> 44.8, pack 59.6 -> 62.2).  Where the V rows are whole 128-byte
// lines apart (slots a multiple of 64) 64 slots write whole lines and 32 half
// ones, which costs more than the split gives from kLineSlots on once the
// output is not in a cache.  Eight workspaces in turn, 32 / 64 slots: gather of
// 3072 190.6 / 169.6 us, 3584 212.1 / 192.6, 4096 239.6 / 215.4, pack 216.8 /
// 197.3, 248.1 / 227.9, 281.0 / 259.9, but 1664 103.6 / 108.1 and 3296 195.9 /
// 195.1, 227.6 / 238.9; one workspace 16.0 / 16.4, 19.3 / 18.9, 21.5 / 21.8.
// Bound by HBM: at 6560 slots the pack moves 269 MB (161 MB written), the
// gather 215 MB (107 MB written).  The packed V and mask leave through
// streaming stores, K through the caches, because the times say so; the bytes
// behind the L2 are the same with V and mask stored through the caches too
// (pack 51.5 and 51.6 thousand KiB fetched), so what it changes lies in the
// MALL, which has no counter.  us, all cached / all streamed / as here: 6560
// slots, three workspaces in turn: pack with its union 68.2 / 59.8 / 59.6,
// gather 45.9 / 43.5 / 41.6; one workspace over 30 pools: pack 49.6 / 52.1 /
// 48.3, gather 37.9 / 41.4 / 37.9 (there the gather gains nothing); a 64-query
// pack of 1664 slots with its union 17.9 / 17.6 / 16.7.  (With streaming loads
// of the rows too: pack with its union 76.3, gather 44.5.)
constexpr uint32_t kShortSlots = 256 * 8 / 32 * 64, kLineSlots = 2560;
inline uint32_t pack_slots(uint32_t count) {
    return count <= kShortSlots && (count < kLineSlots || count % 64 != 0) ? 32u : 64u;
}
template <bool kPack, uint32_t kSlots>
__global__ void __launch_bounds__(kSlots * 4)
pack_kernel(PoolSource ps, MapSource ms, const uint64_t* __restrict__ positions, uint32_t nq,
            uint32_t count, uint16_t* __restrict__ k_out, uint16_t* __restrict__ v_out,
            float* __restrict__ mask, hs_status_t* __restrict__ status, uint32_t stamp) {
    constexpr uint32_t kT = kSlots * 4;
    static_assert(kSlots <= 64 && kSlots % 8 == 0, "one wave looks the slots up");
    __shared__ uint4 vtile[kSlots][17];  // kSlots x 256 B V half row (+pad)
    __shared__ const uint8_t* src_row[kSlots];
    __shared__ uint32_t slot_id[kSlots], slot_ok[kSlots];
    const uint32_t h = blockIdx.y, kv = h >> 2, s0 = blockIdx.x * kSlots, tid = threadIdx.x;

    if (tid < kSlots) {  // wave 0
        const uint32_t s = s0 + tid;
        const uint8_t* src = nullptr;
        uint32_t id = 0xffffffffu;
        int err = HS_OK;  // this lane's first error
        auto fail = [&](int code) { err = err != HS_OK ? err : code; };
        // gqa_pack.hpp:29: positions.back() < 66048; ids beyond it are future.
        uint64_t extent = 0;
        if (kPack) {
            const uint64_t last = positions[nq - 1];
            if (last >= kMaxVisible) fail(HS_ERR_ARGUMENT);
            else extent = last + 1;
        }
        if (s < count) {
            if (kPack) {
                const uint32_t len = ps.lens[h];
                if (len == 0 || len > count) {
                    fail(HS_ERR_ARGUMENT);
                } else if (s < len) {
                    id = ps.ids[static_cast<size_t>(h) * ps.ids_stride + s];
                    int32_t row = -1;
                    if (id < extent && id < ps.max_id)
                        row = ps.row_of_id ? ps.row_of_id[id] : static_cast<int32_t>(id);
                    if (row < 0 || static_cast<uint32_t>(row) >= ps.pool_rows) {
                        fail(HS_ERR_MISSING);
                        id = 0xffffffffu;
                    } else {
                        src = ps.pool + static_cast<size_t>(row) * ps.row_bytes;
                    }
                }
            } else {
                const int32_t row = ms.map[static_cast<size_t>(h) * count + s];
                const int64_t miss = -2 - static_cast<int64_t>(row);
                if (row >= 0 && static_cast<uint32_t>(row) < ms.prefetched_rows && ms.prefetched)
                    src = reinterpret_cast<const uint8_t*>(ms.prefetched) +
                          static_cast<size_t>(row) * 4096;
                else if (row <= -2 && miss < static_cast<int64_t>(ms.miss_rows) && ms.misses)
                    src = reinterpret_cast<const uint8_t*>(ms.misses) +
                          static_cast<size_t>(miss) * 4096;
                else if (row != -1)  // gqa_prefetch_cuda.cu:69 refuses rows beyond the payload
                    fail(HS_ERR_MISSING);
            }
        }
        // a slot with no row reads the fallback row (discarded) so that every
        // load below can be issued unconditionally
        src_row[tid] = src ? src : fallback_row(ps, ms, kPack);
        slot_ok[tid] = src != nullptr;
        slot_id[tid] = id;
        // the workgroup's first error (lowest slot), published by lane 0
        const uint64_t failing = __ballot(err != HS_OK);
        const int first = failing ? __shfl(err, __ffsll(static_cast<long long>(failing)) - 1) : HS_OK;
        if (tid == 0) publish_stamped(status, stamp, first, blockIdx.x == 0 && blockIdx.y == 0);
    }
    __syncthreads();
    // K rows: kSlots x 16 x 16 B; V half rows staged for the transpose.
    // (prefetched and miss rows are 4096 B records: V 2048 B after K)
    const int64_t v_delta = kPack ? ps.v_delta : 2048;
    // Every K and V chunk of the thread's 4 (slot, chunk) pairs is requested
    // before any is stored.  The row pointers come back from LDS without
    // their address space: they are read through global pointers (flat loads
    // can only be waited for all at once).  With no source at all (every
    // slot empty) nothing is read.
    using GlobalU32 = const __attribute__((address_space(1))) uint32_t;
    constexpr uint32_t kPairs = kSlots * 16 / kT;
    uint4 kw[kPairs], vw[kPairs];
    if (fallback_row(ps, ms, kPack) != nullptr) {
#pragma unroll
        for (uint32_t u = 0; u < kPairs; ++u) {
            const uint32_t i = tid + kT * u, s = i >> 4, c = i & 15u;
            const uint8_t* src = src_row[s];
            GlobalU32* kp = (GlobalU32*)(src + kv * 256) + 4 * c;
            GlobalU32* vp = (GlobalU32*)(src + v_delta + kv * 256) + 4 * c;
            kw[u] = make_uint4(kp[0], kp[1], kp[2], kp[3]);
            vw[u] = make_uint4(vp[0], vp[1], vp[2], vp[3]);
        }
    } else {
#pragma unroll
        for (uint32_t u = 0; u < kPairs; ++u) kw[u] = vw[u] = make_uint4(0, 0, 0, 0);
    }
#pragma unroll
    for (uint32_t u = 0; u < kPairs; ++u) {
        const uint32_t i = tid + kT * u, s = i >> 4, c = i & 15u;
        const bool ok = slot_ok[s] != 0;
        vtile[s][c] = ok ? vw[u] : make_uint4(0, 0, 0, 0);
        if (s0 + s < count)
            reinterpret_cast<uint4*>(k_out + (static_cast<size_t>(s0 + s) * 32 + h) * 128)[c] =
                ok ? kw[u] : make_uint4(0, 0, 0, 0);
    }
    __syncthreads();
    // V[h][d][s]: 128 channel rows x kSlots.  A thread gathers 8
    // consecutive slots of one channel from the tile and stores them as one
    // 16-byte word (kSlots / 8 threads cover a channel row); rows whose start
    // is not 16-byte aligned (count % 8 != 0) or that end inside the group
    // store element by element.
    const uint16_t* vt = reinterpret_cast<const uint16_t*>(&vtile[0][0]);
    const bool wide = (count & 7u) == 0 && (reinterpret_cast<uintptr_t>(v_out) & 15u) == 0;
    constexpr uint32_t kRuns = kSlots / 8;
    for (uint32_t i = tid; i < 128 * kRuns; i += kT) {
        const uint32_t d = i / kRuns, sg = (i % kRuns) * 8;
        uint32_t w[4];
#pragma unroll
        for (uint32_t j = 0; j < 4; ++j)
            w[j] = uint32_t(vt[(sg + 2 * j) * (17 * 8) + d]) |
                   (uint32_t(vt[(sg + 2 * j + 1) * (17 * 8) + d]) << 16);
        uint16_t* dst = v_out + (static_cast<size_t>(h) * 128 + d) * count + s0 + sg;
        if (wide && s0 + sg + 8 <= count) {
            store_streaming(dst, make_uint4(w[0], w[1], w[2], w[3]));
        } else {
#pragma unroll
            for (uint32_t j = 0; j < 8; ++j)
                if (s0 + sg + j < count) dst[j] = static_cast<uint16_t>(w[j >> 1] >> ((j & 1u) * 16u));
        }
    }
    if (kPack) {
        // mask rows, 4 slots (16 B) per thread where the row allows
        const uint32_t qpad = (nq + 63) / 64 * 64;
        const bool wide_mask = (count & 3u) == 0 && (reinterpret_cast<uintptr_t>(mask) & 15u) == 0;
        constexpr uint32_t kQuads = kSlots / 4;
        for (uint32_t i = tid; i < qpad * kQuads; i += kT) {
            const uint32_t qi = i / kQuads, sg = (i % kQuads) * 4;
            const uint64_t pos = qi < nq ? positions[qi] : 0;
            uint32_t m[4];  // 0 or -inf
#pragma unroll
            for (uint32_t j = 0; j < 4; ++j) {
                const uint32_t id = slot_id[sg + j];
                const bool open = id != 0xffffffffu && qi < nq && id <= pos;
                m[j] = open ? 0u : 0xff800000u;
            }
            float* dst = mask + (static_cast<size_t>(h) * qpad + qi) * count + s0 + sg;
            if (wide_mask && s0 + sg + 4 <= count) {
                store_streaming(dst, make_uint4(m[0], m[1], m[2], m[3]));
            } else {
#pragma unroll
                for (uint32_t j = 0; j < 4; ++j)
                    if (s0 + sg + j < count) dst[j] = __uint_as_float(m[j]);
            }
        }
    }
}

}  // namespace
}  // namespace hs

extern "C" {

size_t hs_gqa_union_workspace_bytes(uint32_t visible) {
    const size_t v = visible ? visible : 1;
    return hs::align256((v + 31) / 32 * 32 * 4) + hs::align256(32 * 4);
}

int hs_gqa_physical_union(const uint32_t* ids_dev, const uint32_t* lens_dev, size_t ids_stride,
                          uint32_t visible, uint32_t* out_dev, uint32_t* out_n_dev,
                          hs_status_t* status_dev, void* workspace_dev, void* stream) {
    hs::clear_error();
    if (!ids_dev || !lens_dev || !out_dev || !out_n_dev || !status_dev || !workspace_dev)
        return hs::reject("GQA union: null pointer");
    if (visible == 0 || visible > hs::kMaxVisible) return hs::reject("GQA union bounds");
    if (ids_stride > 0xffffffffu) return hs::reject("GQA union: ids_stride too large");
    hipStream_t s = hs::as_stream(stream);
    const uint32_t words = (visible + 31) / 32;
    uint32_t* bitmaps = static_cast<uint32_t*>(workspace_dev);  // [32][words]
    uint32_t* bad_heads = reinterpret_cast<uint32_t*>(static_cast<char*>(workspace_dev) +
                                                      hs::align256(size_t(words) * 32 * 4));
    hipLaunchKernelGGL(hs::union_mark_kernel, dim3(32), dim3(hs::kUnionThreads), 0, s, ids_dev,
                       lens_dev, static_cast<uint32_t>(ids_stride), visible, bitmaps, bad_heads);
    hipLaunchKernelGGL(hs::union_write_kernel, dim3((words + hs::kUnionWords - 1) / hs::kUnionWords),
                       dim3(hs::kUnionThreads), 0, s, bitmaps, bad_heads, visible, out_dev,
                       out_n_dev, status_dev);
    const hipError_t st = hipGetLastError();
    return st == hipSuccess ? HS_OK : hs::hip_fail(st, "union launch");
}

int hs_gqa_pack(const uint8_t* k_pool_dev, const uint8_t* v_pool_dev, size_t row_bytes,
                uint32_t pool_rows, const int32_t* row_of_id_dev, uint32_t max_id,
                const uint32_t* ids_dev, const uint32_t* lens_dev, size_t ids_stride,
                const uint64_t* positions_dev, uint32_t nq, uint32_t count, uint16_t* k_dev,
                uint16_t* v_dev, float* mask_dev, hs_status_t* status_dev, void* stream) {
    hs::clear_error();
    if (!k_pool_dev || !v_pool_dev || !ids_dev || !lens_dev || !positions_dev || !k_dev ||
        !v_dev || !mask_dev || !status_dev)
        return hs::reject("GQA packing: null pointer");
    if (reinterpret_cast<uintptr_t>(status_dev) & 7u)
        return hs::reject("GQA packing: status must be 8-byte aligned");
    if (nq == 0 || nq > 256 || count == 0 || count > hs::kMaxVisible)
        return hs::reject("GQA packing shape");
    if (ids_stride > 0xffffffffu) return hs::reject("GQA packing: ids_stride too large");
    if ((reinterpret_cast<uintptr_t>(k_pool_dev) | reinterpret_cast<uintptr_t>(v_pool_dev)) & 15u)
        return hs::reject("GQA packing: pool alignment");
    if (row_bytes < 2048 || row_bytes % 16 != 0 || row_bytes > (1u << 20))
        return hs::reject("GQA packing: row_bytes must be 2048..1 MiB and a multiple of 16");
    hipStream_t s = hs::as_stream(stream);
    // extent = positions[nq-1] + 1 is read on the device; bound it by max_id.
    const int64_t v_delta =
        reinterpret_cast<intptr_t>(v_pool_dev) - reinterpret_cast<intptr_t>(k_pool_dev);
    hs::PoolSource ps{k_pool_dev, pool_rows, static_cast<uint32_t>(row_bytes), v_delta,
                      row_of_id_dev, max_id, ids_dev, lens_dev, static_cast<uint32_t>(ids_stride)};
    hs::MapSource ms{nullptr, nullptr, nullptr};
    hs::clear_status_if_captured(status_dev, 1, s);
    const uint32_t slots = hs::pack_slots(count);
    hipLaunchKernelGGL((slots == 32 ? hs::pack_kernel<true, 32> : hs::pack_kernel<true, 64>),
                       dim3((count + slots - 1) / slots, 32), dim3(slots * 4), 0, s, ps, ms,
                       positions_dev, nq, count, k_dev, v_dev, mask_dev, status_dev, hs::next_stamp());
    const hipError_t st = hipGetLastError();
    return st == hipSuccess ? HS_OK : hs::hip_fail(st, "pack launch");
}

int hs_gqa_gather_rows(const uint16_t* prefetched_dev, uint32_t prefetched_rows,
                       const uint16_t* misses_dev, uint32_t miss_rows, const int32_t* map_dev,
                       uint32_t count, uint16_t* k_dev, uint16_t* v_dev, hs_status_t* status_dev,
                       void* stream) {
    hs::clear_error();
    if (!map_dev || !k_dev || !v_dev || !status_dev) return hs::reject("gather: null pointer");
    if (reinterpret_cast<uintptr_t>(status_dev) & 7u)
        return hs::reject("gather: status must be 8-byte aligned");
    if (count == 0 || count > hs::kMaxVisible) return hs::reject("gather: count out of range");
    hs::PoolSource ps{};
    hs::MapSource ms{prefetched_dev, misses_dev, map_dev, prefetched_rows, miss_rows};
    hipStream_t s = hs::as_stream(stream);
    hs::clear_status_if_captured(status_dev, 1, s);
    const uint32_t slots = hs::pack_slots(count);
    hipLaunchKernelGGL((slots == 32 ? hs::pack_kernel<false, 32> : hs::pack_kernel<false, 64>),
                       dim3((count + slots - 1) / slots, 32), dim3(slots * 4), 0, s, ps, ms, nullptr,
                       0u, count, k_dev, v_dev, nullptr, status_dev, hs::next_stamp());
    const hipError_t st = hipGetLastError();
    return st == hipSuccess ? HS_OK : hs::hip_fail(st, "gather launch");
}

}  // extern "C"
