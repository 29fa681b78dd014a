// Stable ray-queue compaction on the GPU.
//
// RayQueue::compact_hits (render/scheduling/ray_queue.h:161-185) and compact_rays (:188-207)
// run as a serial loop over the queue on one host thread in the reference.  Here the queue
// is compacted out of place by two launches:
//   1. count:   each block counts the kept entries of its tile (wave ballot + popcount);
//   2. scatter: each block adds up the counts of the tiles before it, ranks its kept entries
//               (ballots, mbcnt, wave totals in LDS) and moves ray / hit / state records.
// Queues of more than kSumTiles tiles get a launch between them that turns the counts into
// offsets.  Kept entries keep their order.  compact_hits also writes the removed (missed) entries
// after the kept ones, in order; the reference's swap loop leaves that tail permuted, and
// callers only use the hit prefix (they shrink the queue to the returned count).
// Traffic per entry: key read twice (4 B), record read and written once (32 + 16 + S B).
// With 2,048 entries per tile, barriers between its chunks and a record per lane the scatter took
// 17 us for 16,000 rays and 58 us for 921,600 hits with 40-byte states, and the offsets a launch of
// their own (4.7 us); whole frames gained from it: path-traced 128x128 905 -> 782 us, 640x480
// 4,393 -> 4,255, a VCM iteration with 27 compactions 5,073 -> 4,713.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <mutex>

#include "common.h"

namespace imba {
namespace {

constexpr int kBlock = 256;
constexpr int kWaves = kBlock / 64;
// Entries per tile: 512 in queues of up to 2,048 such tiles, so that a small queue has blocks for
// every CU, else 2,048: the tiles' sums of the counts before them cost more than the blocks gain.
// us with 512 / 2,048, compact_hits with 40-byte states (16-byte states and compact_rays cross at
// 0.9 to 1.3M entries too): 65,536 entries 9 / 22, 524,288 21 / 33, 786,432 33 / 37, 1,048,576 44 / 39,
// 2,097,152 103 / 99; compact_rays 7 / 15, 16 / 23, 22 / 28, 33 / 34, 65 / 61.
constexpr int kSmallItems = 2, kLargeItems = 8;
constexpr int kSmallTiles = 2048;
// Tiles up to which every block of the scatter adds up the counts itself: all blocks together read
// tiles^2 counts from L2 (67 MB at 4,096 tiles).  us with the sums / with a launch between the two that
// makes offsets of the counts, 16-byte states, compact_hits and compact_rays: 1,048,576 entries (512
// tiles) 30 / 32 and 19 / 21, 8,388,608 (4,096) 293 / 296 and 165 / 165, 12,582,912 437 / 442 and
// 263 / 257, 16,777,216 585 / 595 and 358 / 351.
constexpr int kSumTiles = 4096;

constexpr int tile_of(int n) {
    return n <= kSmallTiles * kBlock * kSmallItems ? kBlock * kSmallItems : kBlock * kLargeItems;
}
// Most tiles a queue of at most n entries has.
constexpr int max_tiles(int n) {
    const int large = (int)(((long long)n + kBlock * kLargeItems - 1) / (kBlock * kLargeItems));
    const int small = (int)(((long long)n + kBlock * kSmallItems - 1) / (kBlock * kSmallItems));
    const int most_small = small < kSmallTiles ? small : kSmallTiles;
    return large > most_small ? large : most_small;
}

enum { kModeHits = 0, kModeRays = 1 };

struct CompactArgs {
    const float4* rays_in;
    const int4* hits_in;
    const int* states_in;
    int stride_dw;  // state record size in dwords
    int n;               // entries (or, with count_dev, the capacity)
    const int* count_dev;  // device entry count read when the launch runs, or null
    float4* rays_out;
    int4* hits_out;
    int* states_out;
    int* block_counts;   // kept entries per tile (or, with `scanned`, before the tile), the total after them
    bool scanned;
    int* count_out;      // device copy of the total, or null
};

// Entries of this launch: n, or the device count clamped to [0, n].
__device__ __forceinline__ int entries(const CompactArgs& a) {
    return a.count_dev ? min(max(*a.count_dev, 0), a.n) : a.n;
}

template <int MODE>
__device__ __forceinline__ bool kept(const CompactArgs& a, int i) {
    if (MODE == kModeHits) return a.hits_in[i].x >= 0;
    return a.states_in[(size_t)i * a.stride_dw] >= 0;
}

__device__ __forceinline__ int lane_rank(unsigned long long mask) {
    return __builtin_amdgcn_mbcnt_hi((unsigned)(mask >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)mask, 0u));
}

template <int MODE, int ITEMS>
__global__ __launch_bounds__(kBlock) void k_count(CompactArgs a) {
    __shared__ int wave_sum[kWaves];
    const int base = blockIdx.x * kBlock * ITEMS;
    const int n = entries(a);
    int cnt = 0;
#pragma unroll
    for (int it = 0; it < ITEMS; it++) {
        const int i = base + it * kBlock + (int)threadIdx.x;
        const bool f = i < n && kept<MODE>(a, i);
        cnt += __popcll(__ballot(f));
    }
    // every lane of a wave holds the same count
    if ((threadIdx.x & 63) == 0) wave_sum[threadIdx.x >> 6] = cnt;
    __syncthreads();
    if (threadIdx.x == 0) {
        int s = 0;
        for (int w = 0; w < kWaves; w++) s += wave_sum[w];
        a.block_counts[blockIdx.x] = s;
    }
}

// Exclusive scan of nb tile counts in place; the total goes to offs[nb] (and to *count_out when
// given).
__global__ __launch_bounds__(1024) void k_scan_offsets(int* offs, int nb, int* count_out) {
    __shared__ int part[1024];
    const int t = threadIdx.x;
    const int per = (nb + 1023) / 1024;
    const int b0 = min(nb, t * per);
    const int b1 = min(nb, b0 + per);
    int s = 0;
    for (int b = b0; b < b1; b++) s += offs[b];
    part[t] = s;
    __syncthreads();
    for (int d = 1; d < 1024; d <<= 1) {
        const int v = t >= d ? part[t - d] : 0;
        __syncthreads();
        part[t] += v;
        __syncthreads();
    }
    int run = part[t] - s;  // exclusive prefix of this thread's chunk
    for (int b = b0; b < b1; b++) {
        const int c = offs[b];
        offs[b] = run;
        run += c;
    }
    if (t == 1023) {
        offs[nb] = part[1023];
        if (count_out) *count_out = part[1023];
    }
}

// Moves the records of the wave's 64 entries from `first` whose bit is set in `mask` to consecutive
// places from `dst`: rays and hits a record per lane; states a unit (4, 8 or 16 bytes) per
// lane, so that neighbouring lanes read and write neighbouring memory (a 40-byte state copied by
// its own lane takes ten instructions that touch every line of the wave's 2.5 KB each).
// `list` holds 64 bytes of the wave's LDS.
template <int MODE, typename UNIT>
__device__ __forceinline__ void move_records(const CompactArgs& a, int first, unsigned long long mask, int dst,
                                             uint8_t* list) {
    const int lane = threadIdx.x & 63;
    const int rank = lane_rank(mask);
    if ((mask >> lane) & 1) {
        const int src = first + lane, to = dst + rank;
        const float4 r0 = a.rays_in[2 * (size_t)src], r1 = a.rays_in[2 * (size_t)src + 1];
        a.rays_out[2 * (size_t)to] = r0;
        a.rays_out[2 * (size_t)to + 1] = r1;
        if (MODE == kModeHits) a.hits_out[to] = a.hits_in[src];
        list[rank] = (uint8_t)lane;
    }
    // the wave's own LDS writes are visible to its later reads
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    const uint32_t per = (uint32_t)a.stride_dw * 4 / (uint32_t)sizeof(UNIT);  // units per state
    const uint32_t units = (uint32_t)__popcll(mask) * per;
    const UNIT* in = reinterpret_cast<const UNIT*>(a.states_in) + (size_t)first * per;
    UNIT* out = reinterpret_cast<UNIT*>(a.states_out) + (size_t)dst * per;
    uint32_t r = (uint32_t)lane / per, w = (uint32_t)lane % per;  // record and unit of this lane
    const uint32_t dr = 64 / per, dw = 64 % per;
    for (uint32_t u = lane; u < units; u += 64) {
        out[u] = in[list[r] * per + w];
        r += dr;
        w += dw;
        if (w >= per) { w -= per; r++; }
    }
    __builtin_amdgcn_wave_barrier();  // the list is reused
}

template <int MODE, int ITEMS, typename UNIT>
__global__ __launch_bounds__(kBlock) void k_scatter(CompactArgs a, int nblocks) {
    __shared__ int wave_cnt[ITEMS][kWaves];
    __shared__ int sums[2][kWaves];
    __shared__ uint8_t lists[kWaves][64];
    const int tile = kBlock * ITEMS;
    const int base = blockIdx.x * tile;
    const int n = entries(a);
    if (base >= n && blockIdx.x > 0) return;
    const int lane = threadIdx.x & 63;
    const int wave = threadIdx.x >> 6;
    unsigned long long m[ITEMS];
#pragma unroll
    for (int it = 0; it < ITEMS; it++) {
        const int i = base + it * kBlock + (int)threadIdx.x;
        m[it] = __ballot(i < n && kept<MODE>(a, i));
        if (lane == 0) wave_cnt[it][wave] = __popcll(m[it]);
    }
    int before = 0, total = 0;  // kept entries before this tile, and in all
    if (a.scanned) {
        before = a.block_counts[blockIdx.x];
        total = a.block_counts[nblocks];
        __syncthreads();
    } else {
        const int live = min(nblocks, (n + tile - 1) / tile);
        for (int b = threadIdx.x; b < live; b += kBlock) {
            const int c = a.block_counts[b];
            total += c;
            before += b < (int)blockIdx.x ? c : 0;
        }
        for (int o = 32; o > 0; o >>= 1) {
            before += __shfl_down(before, o, 64);
            total += __shfl_down(total, o, 64);
        }
        if (lane == 0) {
            sums[0][wave] = before;
            sums[1][wave] = total;
        }
        __syncthreads();
        before = total = 0;
        for (int w = 0; w < kWaves; w++) {
            before += sums[0][w];
            total += sums[1][w];
        }
        if (blockIdx.x == 0 && threadIdx.x == 0) {
            a.block_counts[nblocks] = total;
            if (a.count_out) *a.count_out = total;
        }
    }
    int removed = base - before;  // removed entries before this tile
#pragma unroll
    for (int it = 0; it < ITEMS; it++) {
        int wave_kept = 0, chunk_kept = 0;  // in the waves before this one, and in the chunk
#pragma unroll
        for (int w = 0; w < kWaves; w++) {
            const int c = wave_cnt[it][w];
            wave_kept += w < wave ? c : 0;
            chunk_kept += c;
        }
        const int first = base + it * kBlock + wave * 64;
        if (first < n) {
            move_records<MODE, UNIT>(a, first, m[it], before + wave_kept, lists[wave]);
            if (MODE == kModeHits) {
                const unsigned long long valid = n - first >= 64 ? ~0ull : ~(~0ull << (n - first));
                const int dst = total + removed + wave * 64 - wave_kept;
                move_records<MODE, UNIT>(a, first, valid & ~m[it], dst, lists[wave]);
            }
        }
        before += chunk_kept;
        removed += kBlock - chunk_kept;  // (only the last chunk is partial)
    }
}

// The launches of one compaction of a.n entries at most; states in the widest unit that their
// size and addresses allow.
template <int MODE, int ITEMS>
void launch_compact(CompactArgs a, int nb, hipStream_t s) {
    a.scanned = nb > kSumTiles;
    hipLaunchKernelGGL((k_count<MODE, ITEMS>), dim3(nb), dim3(kBlock), 0, s, a);
    if (a.scanned)
        hipLaunchKernelGGL(k_scan_offsets, dim3(1), dim3(1024), 0, s, a.block_counts, nb, a.count_out);
    const uintptr_t bits = (uintptr_t)a.states_in | (uintptr_t)a.states_out | (uintptr_t)(a.stride_dw * 4);
    if (bits % 16 == 0)
        hipLaunchKernelGGL((k_scatter<MODE, ITEMS, uint4>), dim3(nb), dim3(kBlock), 0, s, a, nb);
    else if (bits % 8 == 0)
        hipLaunchKernelGGL((k_scatter<MODE, ITEMS, uint2>), dim3(nb), dim3(kBlock), 0, s, a, nb);
    else
        hipLaunchKernelGGL((k_scatter<MODE, ITEMS, uint32_t>), dim3(nb), dim3(kBlock), 0, s, a, nb);
}
template <int MODE>
int launch_compact(const CompactArgs& a, hipStream_t s) {
    const int tile = tile_of(a.n), nb = std::max(1, ceil_div(a.n, tile));
    if (tile == kBlock * kSmallItems) launch_compact<MODE, kSmallItems>(a, nb, s);
    else launch_compact<MODE, kLargeItems>(a, nb, s);
    IMBA_HIP_TRY(hipGetLastError());
    return IMBA_OK;
}

thread_local Scratch t_offsets[64];

// Block offsets of the allocation-free compaction (imba_compact_hits_noalloc): one array per
// device for the life of the process, kNoAllocMaxBlocks + 1 ints (256 KiB + 4 B), enough for
// 134,217,728 entries.  Host code never passes this name to a kernel (on the host it is only a
// stand-in for the symbol); it uses the device address hipGetSymbolAddress gave for the
// current device.
constexpr int kNoAllocMaxBlocks = 65536;
static_assert((long long)kNoAllocMaxBlocks * kBlock * kLargeItems == IMBA_COMPACT_NOALLOC_MAX_COUNT, "header limit");
static_assert(kNoAllocMaxBlocks >= kSmallTiles, "tiles of small queues");
static __device__ __align__(256) int scratch[kNoAllocMaxBlocks + 1];

constexpr int kMaxDevices = 64;
std::mutex g_scratch_mu;
int* g_scratch_ptr[kMaxDevices] = {};

// The current device's copy of `scratch`, looked up once per device.
int scratch_for_device(int dev, int** out) {
    if (dev < 0 || dev >= kMaxDevices) return fail(IMBA_ERR_INVALID_ARG, "device %d out of range", dev);
    std::lock_guard<std::mutex> lk(g_scratch_mu);
    if (!g_scratch_ptr[dev]) {
        void* p = nullptr;
        IMBA_HIP_TRY(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
        if (!p) return fail(IMBA_ERR_HIP, "hipGetSymbolAddress returned no address for the compaction scratch");
        g_scratch_ptr[dev] = (int*)p;
    }
    *out = g_scratch_ptr[dev];
    return IMBA_OK;
}

template <int MODE>
int run_compact(CompactArgs a, int* new_count, void* stream, bool static_scratch = false) {
    if (a.n < 0) return fail(IMBA_ERR_INVALID_ARG, "count < 0");
    if (a.stride_dw <= 0) return fail(IMBA_ERR_INVALID_ARG, "state stride must be a positive multiple of 4 bytes");
    if (static_scratch && a.n > IMBA_COMPACT_NOALLOC_MAX_COUNT)
        return fail(IMBA_ERR_CAPACITY, "count %d exceeds the %d entries of the allocation-free compaction", a.n,
                    IMBA_COMPACT_NOALLOC_MAX_COUNT);
    if (a.n == 0) {
        if (new_count) *new_count = 0;
        return IMBA_OK;
    }
    if (!a.rays_in || !a.states_in || !a.rays_out || !a.states_out || (MODE == kModeHits && (!a.hits_in || !a.hits_out)))
        return fail(IMBA_ERR_INVALID_ARG, "NULL buffer");
    int dev = 0;
    IMBA_HIP_TRY(hipGetDevice(&dev));
    const int nb = ceil_div(a.n, tile_of(a.n));
    if (static_scratch) {
        int r = scratch_for_device(dev, &a.block_counts);
        if (r) return r;
    } else {
        // Room for every smaller queue too (one of 1,048,576 entries has more tiles than a larger
        // one), so that a call that was made once can be recorded with any smaller size.
        Scratch& sc = t_offsets[dev & 63];
        int r = grow_buffer(sc, sizeof(int) * ((size_t)std::max(max_tiles(a.n), kSmallTiles) + 1));
        if (r) return r;
        a.block_counts = (int*)sc.ptr;
    }
    bool sync;
    hipStream_t s;
    if (static_scratch) {
        // no per-thread stream is created here: NULL is the device's null stream
        s = (hipStream_t)stream;
        sync = stream == nullptr;
    } else {
        s = resolve_stream(stream, &sync);
    }
    {
        const int r = launch_compact<MODE>(a, s);
        if (r) return r;
    }
    if (new_count) {
        int total = 0;
        IMBA_HIP_TRY(hipMemcpyAsync(&total, a.block_counts + nb, sizeof(int), hipMemcpyDeviceToHost, s));
        IMBA_HIP_TRY(hipStreamSynchronize(s));
        // compact_rays keeps the size when nothing was removed (ray_queue.h:203-206): the total
        // is then the input count either way.
        *new_count = total;
    } else if (sync) {
        IMBA_HIP_TRY(hipStreamSynchronize(s));
    }
    return IMBA_OK;
}

}  // namespace
}  // namespace imba

using namespace imba;

extern "C" {

size_t imba_compact_workspace_size(int capacity) {
    return sizeof(int) * ((size_t)std::max(1, max_tiles(capacity > 0 ? capacity : 0)) + 1);
}

int imba_compact_rays_dev(const ImbaRay* rays_in, const void* states_in, int state_stride, int capacity,
                          const int* count_dev, ImbaRay* rays_out, void* states_out, int* new_count_dev,
                          void* workspace, void* stream) {
    IMBA_CHECK_ARG(state_stride > 0 && state_stride % 4 == 0, "state_stride must be a positive multiple of 4");
    IMBA_CHECK_ARG(capacity >= 0, "capacity < 0");
    IMBA_CHECK_ARG(count_dev && new_count_dev && workspace, "count_dev, new_count_dev and workspace are required");
    IMBA_CHECK_ARG(capacity == 0 || (rays_in && states_in && rays_out && states_out), "NULL buffer");
    CompactArgs a{};
    a.rays_in = (const float4*)rays_in;
    a.states_in = (const int*)states_in;
    a.stride_dw = state_stride / 4;
    a.n = capacity;
    a.count_dev = count_dev;
    a.rays_out = (float4*)rays_out;
    a.states_out = (int*)states_out;
    a.block_counts = (int*)workspace;
    a.count_out = new_count_dev;
    bool sync;
    hipStream_t s = resolve_stream(stream, &sync);
    const int r = launch_compact<kModeRays>(a, s);
    if (r) return r;
    if (sync) IMBA_HIP_TRY(hipStreamSynchronize(s));
    return IMBA_OK;
}

int imba_compact_hits(const ImbaRay* rays_in, const ImbaHit* hits_in, const void* states_in, int state_stride, int count,
                      ImbaRay* rays_out, ImbaHit* hits_out, void* states_out, int* new_count, void* stream) {
    IMBA_CHECK_ARG(state_stride > 0 && state_stride % 4 == 0, "state_stride must be a positive multiple of 4");
    CompactArgs a{};
    a.rays_in = (const float4*)rays_in;
    a.hits_in = (const int4*)hits_in;
    a.states_in = (const int*)states_in;
    a.stride_dw = state_stride / 4;
    a.n = count;
    a.rays_out = (float4*)rays_out;
    a.hits_out = (int4*)hits_out;
    a.states_out = (int*)states_out;
    return run_compact<kModeHits>(a, new_count, stream);
}

int imba_compact_hits_noalloc(const ImbaRay* rays_in, const ImbaHit* hits_in, const void* states_in, int state_stride,
                              int count, ImbaRay* rays_out, ImbaHit* hits_out, void* states_out, int* new_count,
                              void* stream) {
    IMBA_CHECK_ARG(state_stride > 0 && state_stride % 4 == 0, "state_stride must be a positive multiple of 4");
    CompactArgs a{};
    a.rays_in = (const float4*)rays_in;
    a.hits_in = (const int4*)hits_in;
    a.states_in = (const int*)states_in;
    a.stride_dw = state_stride / 4;
    a.n = count;
    a.rays_out = (float4*)rays_out;
    a.hits_out = (int4*)hits_out;
    a.states_out = (int*)states_out;
    return run_compact<kModeHits>(a, new_count, stream, true);
}


int imba_compact_rays(const ImbaRay* rays_in, const void* states_in, int state_stride, int count, ImbaRay* rays_out,
                      void* states_out, int* new_count, void* stream) {
    IMBA_CHECK_ARG(state_stride > 0 && state_stride % 4 == 0, "state_stride must be a positive multiple of 4");
    CompactArgs a{};
    a.rays_in = (const float4*)rays_in;
    a.states_in = (const int*)states_in;
    a.stride_dw = state_stride / 4;
    a.n = count;
    a.rays_out = (float4*)rays_out;
    a.states_out = (int*)states_out;
    return run_compact<kModeRays>(a, new_count, stream);
}

}  // extern "C"
