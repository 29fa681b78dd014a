// Photon hash grid on the GPU: counting-sort build and k-capped range query.
//
// HashGrid (rangesearch/rangesearch.h:21-158) builds on the host with TBB: bounds reduce,
// atomic count per bucket, serial exclusive scan, atomic scatter.  Here:
//   bounds   k_bounds: per-block min/max
//   keys     k_grid_keys combines the bounds (grown by 0.1%, derived values) and writes the
//            bucket of each photon and the sort's first tile counts
//   sort     stable LSD radix sort of the photon indices by bucket (radix.h): the slot order is by
//            bucket, then by photon index, which is deterministic and equals a serial run of
//            the reference's scatter
//   slots    k_slots: positions copied to slot order as float4 (x, y, z, index bits), and the
//            bounds of the buckets' photons among each 64 slots
//   ends     k_ends: each bucket's end from the sorted keys, an inclusive max-scan carrying it
//            over the empty buckets; it also joins the bounds of buckets that go on past 64 slots
// 4M photons, 8M buckets: 446 us in 26 launches before the sort was rewritten and the smaller
// launches were merged, now 291 in 12.
// The query visits the same 8 buckets in the same order as the reference (duplicates
// included), a wave taking its queries one after the other (two where there are enough), and keeps
// the k-capped, distance-sorted list in lanes 0..k-1 with the reference's insertion rule.  Squared
// distances are computed without fused multiply-add, as on the host.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cfloat>

#include "common.h"
#include "grid_query.h"
#include "grid_size.h"
#include "radix.h"

namespace imba {
namespace {

constexpr int kBoundsBlocks = 512;
constexpr int kBlock = 256;
constexpr int kScanItems = 8;
constexpr int kScanTile = kBlock * kScanItems;
constexpr int kSortItems = 16;  // radix tiles of 4096 entries

__device__ __forceinline__ const float* photon_pos(const unsigned char* base, int stride, int off, int i) {
    return reinterpret_cast<const float*>(base + (size_t)i * stride + off);
}

__device__ __forceinline__ float pick_min(float a, float b) { return a < b ? a : b; }
__device__ __forceinline__ float pick_max(float a, float b) { return a > b ? a : b; }

// Block-wide bounds of the threads' bounds (min / max are exact in any order), in every thread.
__device__ __forceinline__ void block_bounds(float* lo, float* hi) {
    __shared__ float red[6][kBlock / 64];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
#pragma unroll
    for (int k = 0; k < 3; k++) {
        for (int o = 32; o > 0; o >>= 1) {
            lo[k] = pick_min(lo[k], __shfl_xor(lo[k], o, 64));
            hi[k] = pick_max(hi[k], __shfl_xor(hi[k], o, 64));
        }
        if (lane == 0) {
            red[k][wave] = lo[k];
            red[3 + k][wave] = hi[k];
        }
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < 3; k++)
        for (int w = 0; w < kBlock / 64; w++) {
            lo[k] = pick_min(lo[k], red[k][w]);
            hi[k] = pick_max(hi[k], red[3 + k][w]);
        }
}

// Bounds of the photons, one box per block.
__global__ __launch_bounds__(kBlock) void k_bounds(const unsigned char* ph, int stride, int off, int n, float* partial) {
    float lo[3] = {FLT_MAX, FLT_MAX, FLT_MAX}, hi[3] = {-FLT_MAX, -FLT_MAX, -FLT_MAX};
    const int step = gridDim.x * kBlock;
    for (int i = blockIdx.x * kBlock + threadIdx.x; i < n; i += step) {
        const float* p = photon_pos(ph, stride, off, i);
#pragma unroll
        for (int k = 0; k < 3; k++) {
            const float v = p[k];
            lo[k] = pick_min(lo[k], v);
            hi[k] = pick_max(hi[k], v);
        }
    }
    block_bounds(lo, hi);
    if (threadIdx.x < 6) partial[6 * blockIdx.x + threadIdx.x] = threadIdx.x < 3 ? lo[threadIdx.x] : hi[threadIdx.x - 3];
}

// Every block combines the bounds of all (a few KB from L2) into the grid parameters; block 0 stores
// them for the later kernels.  Then the bucket of each photon of the block's tile, and the tile's
// counts of the keys' lowest digit.
__global__ __launch_bounds__(kBlock) void k_grid_keys(const unsigned char* ph, int stride, int off, int n,
                                                      const float* partial, int nparts, GridParams* gp, float radius,
                                                      int table, int* keys, int n_tiles, int* counts) {
    __shared__ RadixTile<kSortItems> tile;
    float lo[3] = {FLT_MAX, FLT_MAX, FLT_MAX}, hi[3] = {-FLT_MAX, -FLT_MAX, -FLT_MAX};
    for (int b = threadIdx.x; b < nparts; b += kBlock)
        for (int k = 0; k < 3; k++) {
            lo[k] = pick_min(lo[k], partial[6 * b + k]);
            hi[k] = pick_max(hi[k], partial[6 * b + 3 + k]);
        }
    block_bounds(lo, hi);
    GridParams g;
    for (int k = 0; k < 3; k++) {
        const float e = hi[k] - lo[k];
        g.bmax[k] = hi[k] + e * 0.001f;
        g.bmin[k] = lo[k] - e * 0.001f;
    }
    g.radius = radius;
    g.radius_sqr = radius * radius;
    g.cell_size = radius * 2.0f;
    g.inv_cell_size = 1.0f / g.cell_size;
    g.table_size = table;
    g.count = n;
    if (blockIdx.x == 0 && threadIdx.x == 0) *gp = g;
    if (n == 0) return;
    tile.clear();
    float p[kSortItems][3];
#pragma unroll
    for (int it = 0; it < kSortItems; it++) {
        const float* q = photon_pos(ph, stride, off, min(tile.index(it), n - 1));
        for (int k = 0; k < 3; k++) p[it][k] = q[k];
    }
#pragma unroll
    for (int it = 0; it < kSortItems; it++) {
        const int i = tile.index(it);
        if (i < n) {
            const int cx = (int)floorf(g.inv_cell_size * (p[it][0] - g.bmin[0]));
            const int cy = (int)floorf(g.inv_cell_size * (p[it][1] - g.bmin[1]));
            const int cz = (int)floorf(g.inv_cell_size * (p[it][2] - g.bmin[2]));
            const int key = bucket_of((uint32_t)cx, (uint32_t)cy, (uint32_t)cz, table);
            keys[i] = key;
            tile.add(key & 255);
        }
    }
    tile.store(counts, n_tiles);
}

// One step of a scan over the wave's runs of equal keys: the bounds of the lane that the DPP control
// names (in the rows of the mask) join this lane's if its key is the same.
template <int CTRL, int ROWS>
__device__ __forceinline__ void join_bounds(int key, uint32_t* lo, uint32_t* hi) {
    const bool same = __builtin_amdgcn_update_dpp(~key, key, CTRL, ROWS, 0xF, false) == key;
#pragma unroll
    for (int a = 0; a < 3; a++) {
        const uint32_t l = (uint32_t)__builtin_amdgcn_update_dpp((int)lo[a], (int)lo[a], CTRL, ROWS, 0xF, false);
        const uint32_t h = (uint32_t)__builtin_amdgcn_update_dpp((int)hi[a], (int)hi[a], CTRL, ROWS, 0xF, false);
        lo[a] = same ? min(lo[a], l) : lo[a];
        hi[a] = same ? max(hi[a], h) : hi[a];
    }
}

// Slot order: the photons' positions, and the bounds of every non-empty bucket's photons (the
// queries skip buckets that lie beyond their limit; an empty bucket's entry is never used), in the
// order-preserving integer form of grid_query.h.  A wave takes 64 consecutive slots at a time and
// reduces the runs of equal keys (the keys are sorted, so equal keys are contiguous) with DPP row
// shifts and broadcasts; a run's last lane stores its bounds.  A run that began before these slots
// leaves them in heads[slot / 64] instead, for k_ends to join.  Bound by the scattered reads of the
// positions (a cache line each; a thread's four are in flight together): 4M photons 91 us.  With
// the boxes cleared here and joined by atomics in a launch of their own it took 92 + 39.
constexpr int kSlotItems = 4;
__global__ __launch_bounds__(kBlock) void k_slots(const unsigned char* ph, int stride, int off, int n, const int* order,
                                                  const int* keys_sorted, float4* pos4, uint32_t* box, uint32_t* heads) {
    const int base = blockIdx.x * kBlock * kSlotItems + (int)threadIdx.x;
    const int lane = threadIdx.x & 63;
    float p[kSlotItems][3];
    int idx[kSlotItems], keys[kSlotItems], before[kSlotItems];
#pragma unroll
    for (int it = 0; it < kSlotItems; it++) {
        const int s = base + it * kBlock;
        idx[it] = order[min(s, n - 1)];
        keys[it] = s < n ? keys_sorted[s] : -1;
        before[it] = s - lane > 0 && s - lane < n ? keys_sorted[s - lane - 1] : -1;  // key before the wave's slots
    }
#pragma unroll
    for (int it = 0; it < kSlotItems; it++) {
        const float* q = photon_pos(ph, stride, off, idx[it]);
        for (int k = 0; k < 3; k++) p[it][k] = q[k];
    }
#pragma unroll
    for (int it = 0; it < kSlotItems; it++) {
        const int s = base + it * kBlock;
        const int key = keys[it];
        uint32_t lo[3], hi[3];
#pragma unroll
        for (int a = 0; a < 3; a++) lo[a] = hi[a] = ordered_bits(p[it][a]);
        join_bounds<0x111, 0xF>(key, lo, hi);  // row_shr:1, 2, 4, 8: the 16 lanes of a row
        join_bounds<0x112, 0xF>(key, lo, hi);
        join_bounds<0x114, 0xF>(key, lo, hi);
        join_bounds<0x118, 0xF>(key, lo, hi);
        join_bounds<0x142, 0xA>(key, lo, hi);  // row_bcast:15: the last lane of rows 0, 2 to rows 1, 3
        join_bounds<0x143, 0xC>(key, lo, hi);  // row_bcast:31: lane 31 to rows 2 and 3
        const int next = __shfl_down(key, 1, 64);
        if (s < n) {
            pos4[s] = make_float4(p[it][0], p[it][1], p[it][2], __int_as_float(idx[it]));
            if (lane == 63 || next != key) {  // the run's last lane (-1 is no key)
                uint2* e = reinterpret_cast<uint2*>(before[it] == key ? heads + 6 * (size_t)(s >> 6)
                                                                      : box + 6 * (size_t)key);
                e[0] = make_uint2(lo[0], lo[1]);
                e[1] = make_uint2(lo[2], hi[0]);
                e[2] = make_uint2(hi[1], hi[2]);
            }
        }
    }
}

// Photons in buckets before `bucket`: the first slot whose key is not less, searched 64 places at a
// time by a wave.
__device__ __forceinline__ int slots_before(const int* keys_sorted, int n, int bucket) {
    const int lane = threadIdx.x & 63;
    int lo = 0, len = n;  // the answer lies in [lo, lo + len]
    while (len > 0) {
        const int step = (len + 63) / 64;
        const int at = lo + lane * step;
        const bool less = at < lo + len && keys_sorted[at] < bucket;
        const int k = __popcll(__ballot(less));  // the first k probes are less
        if (k == 0) return lo;
        const int end = lo + len;
        lo += (k - 1) * step + 1;
        len = min(step - 1, end - lo);
    }
    return lo;
}

// The buckets' ends, 2048 buckets per block: the block finds its slots in the sorted keys, marks slot +
// 1 at the last slot of each bucket in LDS, and an inclusive max-scan from the slots before carries it
// over the empty buckets.  Where the block's buckets hold many slots each bucket's end is searched
// instead, so that a crowded bucket costs the steps of a search and not a walk (the line lies at 64 slots
// a thread, well above the 1/2 a bucket that the table's size gives).  4M photons, 8M buckets: 34 us;
// with the ends cleared and marked in memory by the launches before, the scan took 28 and the launch
// that cleared them 5 more.
constexpr int kManySlots = 8 * kScanTile;
__global__ __launch_bounds__(kBlock) void k_ends(int* ends, int table, const int* keys_sorted, int n,
                                                 const uint32_t* heads, uint32_t* box) {
    __shared__ int range[kBlock / 64];
    __shared__ __attribute__((aligned(16))) int mark[kScanTile];
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    const int base = blockIdx.x * kScanTile;
    // The runs that go on past 64 slots (table >= 2 n, so the grid has n / 64 threads).
    const long long begin = 64ll * ((int)blockIdx.x * kBlock + t);
    if (begin > 0 && begin < n) {
        const int key = keys_sorted[begin];
        if (keys_sorted[begin - 1] == key) {
            const uint32_t* h = heads + 6 * (begin >> 6);
            uint32_t* e = box + 6 * (size_t)key;
            for (int a = 0; a < 3; a++) {
                atomicMin(e + a, h[a]);
                atomicMax(e + 3 + a, h[3 + a]);
            }
        }
    }
    if (wave < 2) {
        const int r = slots_before(keys_sorted, n, wave == 0 ? base : min(table, base + kScanTile));
        if (lane == 0) range[wave] = r;
    }
    int4* mark4 = reinterpret_cast<int4*>(mark);
    for (int i = t; i < kScanTile / 4; i += kBlock) mark4[i] = make_int4(0, 0, 0, 0);
    __syncthreads();
    const int lo = range[0], hi = range[1];
    __syncthreads();
    int x[kScanItems];
    if (hi - lo <= kManySlots) {
        for (int s = lo + t; s < hi; s += kBlock) {
            const int key = keys_sorted[s];
            if (s == n - 1 || keys_sorted[s + 1] != key) mark[key - base] = s + 1;
        }
        __syncthreads();
#pragma unroll
        for (int k = 0; k < kScanItems; k += 4) {
            const int4 m = mark4[(t * kScanItems + k) / 4];
            x[k] = m.x, x[k + 1] = m.y, x[k + 2] = m.z, x[k + 3] = m.w;
        }
    } else {  // the first slot after the bucket, by halving, the thread's buckets side by side
#pragma unroll
        for (int k = 0; k < kScanItems; k++) x[k] = lo;
        for (int step = 1 << (31 - __clz(hi - lo)); step > 0; step >>= 1)
#pragma unroll
            for (int k = 0; k < kScanItems; k++)
                if (x[k] + step <= hi && keys_sorted[x[k] + step - 1] <= base + t * kScanItems + k) x[k] += step;
    }
#pragma unroll
    for (int k = 1; k < kScanItems; k++) x[k] = max(x[k], x[k - 1]);
    int run = x[kScanItems - 1];
    for (int o = 1; o < 64; o <<= 1) {
        const int y = __shfl_up(run, o, 64);
        if (lane >= o) run = max(run, y);
    }
    if (lane == 63) range[wave] = run;
    const int up = __shfl_up(run, 1, 64);
    run = max(lo, lane > 0 ? up : 0);
    __syncthreads();
    for (int w = 0; w < wave; w++) run = max(run, range[w]);
    const int first = base + t * kScanItems;
#pragma unroll
    for (int k = 0; k < kScanItems; k++) x[k] = max(x[k], run);
    if (first + kScanItems <= table) {
#pragma unroll
        for (int k = 0; k < kScanItems; k += 4)
            *reinterpret_cast<int4*>(ends + first + k) = make_int4(x[k], x[k + 1], x[k + 2], x[k + 3]);
    } else {
#pragma unroll
        for (int k = 0; k < kScanItems; k++)
            if (first + k < table) ends[first + k] = x[k];
    }
}

// `per` queries per wave (query_wave_list); the lists go to out_idx / out_dist.
__global__ __launch_bounds__(kBlock) void k_query_wave(const GridParams* gp, const int* ends, const float4* pos4,
                                                       const uint32_t* box, const unsigned char* qs, int qstride,
                                                       int qoff, int nq, int per, int k, int* out_idx, float* out_dist,
                                                       int* out_count) {
    const int lane = (int)(threadIdx.x & 63);
    const int q0 = (blockIdx.x * (kBlock / 64) + (int)(threadIdx.x >> 6)) * per;
    const int n = min(per, nq - q0);
    if (n <= 0) return;  // whole waves leave together
    const GridParams g = *gp;
    const float* qp = photon_pos(qs, qstride, qoff, q0 + min(lane >> 3, n - 1));
    const float x = qp[0], y = qp[1], z = qp[2];
    const GridProbes probes = grid_probes(g, ends, box, x, y, z, (lane >> 3) < n);
    for (int i = 0; i < n; i++) {
        float my_dist;
        int my_idx;
        const int count = query_wave_list<false>(g, pos4, probes, 8 * i, lane_value(x, 8 * i), lane_value(y, 8 * i),
                                                 lane_value(z, 8 * i), k, my_dist, my_idx);
        const size_t q = (size_t)(q0 + i);
        if (lane < count) {
            out_idx[q * k + lane] = my_idx;
            if (out_dist) out_dist[q * k + lane] = my_dist;
        }
        if (lane == 0) out_count[q] = count;
    }
}

// k > 64: the same scan and insertion rule with the k-capped list in LDS, one query per wave
// and one wave per block (dynamic LDS: k distances, then k photon indices).  Inserting at
// position pos moves the entries [pos, count - 1) one slot up, 64 at a time from the top: the
// wave reads 64 entries, then writes them one slot higher, so every entry is read before it is
// overwritten.  The insertion position is the number of entries <= the candidate, counted over
// the list by all lanes.
constexpr int kQueryMaxK = 4096;

__global__ __launch_bounds__(64) void k_query_lds(const GridParams* gp, const int* ends, const float4* pos4,
                                                  const unsigned char* qs, int qstride, int qoff, int nq, int k,
                                                  int* out_idx, float* out_dist, int* out_count) {
    extern __shared__ float list_lds[];
    float* ld = list_lds;
    int* li = reinterpret_cast<int*>(list_lds + k);
    const int q = blockIdx.x;
    if (q >= nq) return;
    const int lane = (int)threadIdx.x;
    const float* qp = photon_pos(qs, qstride, qoff, q);
    const float qx = qp[0], qy = qp[1], qz = qp[2];
    const GridParams g = *gp;
    int count = 0;
    const bool inside = qx >= g.bmin[0] && qy >= g.bmin[1] && qz >= g.bmin[2] &&
                        qx <= g.bmax[0] && qy <= g.bmax[1] && qz <= g.bmax[2];
    if (inside && g.count > 0) {
        const float cx = g.inv_cell_size * (qx - g.bmin[0]);
        const float cy = g.inv_cell_size * (qy - g.bmin[1]);
        const float cz = g.inv_cell_size * (qz - g.bmin[2]);
        const float fx = floorf(cx), fy = floorf(cy), fz = floorf(cz);
        const int px = (int)fx, py = (int)fy, pz = (int)fz;
        const int pxo = px + ((cx - fx) < 0.5f ? -1 : 1);
        const int pyo = py + ((cy - fy) < 0.5f ? -1 : 1);
        const int pzo = pz + ((cz - fz) < 0.5f ? -1 : 1);
        int begin = 0, size = 0;
        if (lane < 8) {
            const int x = (lane & 4) ? pxo : px;
            const int y = (lane & 2) ? pyo : py;
            const int z = (lane & 1) ? pzo : pz;
            const int b = bucket_of((uint32_t)x, (uint32_t)y, (uint32_t)z, g.table_size);
            begin = b == 0 ? 0 : ends[b - 1];
            size = ends[b] - begin;
        }
        int pre = size;
        for (int o = 1; o < 8; o <<= 1) {
            const int y = __shfl_up(pre, o, 64);
            if (lane >= o) pre += y;
        }
        pre -= size;
        int beg_j[8], pre_j[8];
#pragma unroll
        for (int j = 0; j < 8; j++) {
            beg_j[j] = __builtin_amdgcn_readlane(begin, j);
            pre_j[j] = __builtin_amdgcn_readlane(pre, j);
        }
        const int total = __builtin_amdgcn_readlane(pre + size, 7);
        float kth = 0.0f;
        for (int base = 0; base < total; base += 64) {
            const int c = base + lane;
            const bool valid = c < total;
            float d2 = 0.0f;
            int pid = -1;
            if (valid) {
                int slot = 0;
#pragma unroll
                for (int j = 0; j < 8; j++)
                    if (c >= pre_j[j]) slot = beg_j[j] + (c - pre_j[j]);
                const float4 p = pos4[slot];
                const float dx = qx - p.x, dy = qy - p.y, dz = qz - p.z;
                d2 = dx * dx + dy * dy + dz * dz;
                pid = __float_as_int(p.w);
            }
            const float lim = count == k ? kth : g.radius_sqr;
            unsigned long long m = __ballot(valid && d2 <= lim && d2 <= g.radius_sqr);
            while (m) {
                const int src = __builtin_ctzll(m);
                m &= m - 1;
                const float dd = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(d2), src));
                const int id = __builtin_amdgcn_readlane(pid, src);
                if (count == k) {
                    if (kth < dd) continue;
                } else {
                    count++;
                }
                const int keep = count - 1;  // entries that stay (the last one drops when full)
                int le = 0;
                for (int j = lane; j < keep; j += 64) le += ld[j] <= dd ? 1 : 0;
                for (int o = 32; o > 0; o >>= 1) le += __shfl_xor(le, o, 64);
                const int pos = le;
                for (int top = keep - 1; top >= pos; top -= 64) {
                    const int j = top - lane;
                    const bool act = j >= pos;
                    float v = 0.0f;
                    int w = 0;
                    if (act) {
                        v = ld[j];
                        w = li[j];
                    }
                    __syncthreads();
                    if (act) {
                        ld[j + 1] = v;
                        li[j + 1] = w;
                    }
                    __syncthreads();
                }
                if (lane == 0) {
                    ld[pos] = dd;
                    li[pos] = id;
                }
                __syncthreads();
                if (count == k) kth = ld[k - 1];
            }
        }
    }
    for (int j = lane; j < count; j += 64) {
        out_idx[(size_t)q * k + j] = li[j];
        if (out_dist) out_dist[(size_t)q * k + j] = ld[j];
    }
    if (lane == 0) out_count[q] = count;
}

// A new buffer of `want` elements in place of p, one of those whose capacity is `cap`: zero from
// when the old one is gone.
template <typename T, typename CAP>
int replace(T*& p, CAP& cap, size_t want) {
    if (p) IMBA_HIP_TRY(hipFree(p));
    p = nullptr;
    cap = 0;
    IMBA_HIP_TRY(hipMalloc((void**)&p, sizeof(T) * std::max<size_t>(want, 1)));
    return IMBA_OK;
}

// Buffers for `count` photons and `table` buckets.
int reserve(ImbaHashGrid* g, int count, int table) {
    int r = IMBA_OK;
    if (table > g->table_cap) {
        if ((r = replace(g->cell_ends, g->table_cap, table))) return r;
        if ((r = replace(g->bucket_box, g->table_cap, grid_box_words(table)))) return r;
        g->table_cap = table;
    }
    if (count > g->cap) {
        for (int** p : {&g->order, &g->keys_a, &g->vals_a, &g->keys_b, &g->vals_b})
            if ((r = replace(*p, g->cap, count))) return r;
        if ((r = replace(g->pos4, g->cap, count))) return r;
        g->cap = count;
    }
    const size_t digits = radix_counts_size<kSortItems>(std::max(count, 1));
    if (digits > g->digits_cap) {
        if ((r = replace(g->digits, g->digits_cap, digits))) return r;
        g->digits_cap = digits;
    }
    return IMBA_OK;
}

}  // namespace
}  // namespace imba

using namespace imba;

extern "C" {

int imba_hashgrid_create(ImbaHashGrid** out) {
    IMBA_CHECK_ARG(out, "out is NULL");
    ImbaHashGrid* g = new ImbaHashGrid();
    if (hipGetDevice(&g->device) != hipSuccess) g->device = 0;
    if (hipMalloc((void**)&g->d_params, sizeof(GridParams)) != hipSuccess ||
        hipMalloc((void**)&g->partial, sizeof(float) * 6 * kBoundsBlocks) != hipSuccess) {
        imba_hashgrid_release(g);
        return fail(IMBA_ERR_OUT_OF_MEMORY, "hash grid parameters");
    }
    GridParams zero{};
    if (hipMemcpy(g->d_params, &zero, sizeof(zero), hipMemcpyHostToDevice) != hipSuccess) {
        imba_hashgrid_release(g);
        return fail(IMBA_ERR_HIP, "hash grid parameters");
    }
    *out = g;
    return IMBA_OK;
}

int imba_hashgrid_release(ImbaHashGrid* g) {
    if (!g) return IMBA_OK;
    void* ptrs[] = {g->cell_ends, g->order, g->keys_a, g->vals_a, g->keys_b, g->vals_b, g->pos4, g->d_params,
                    g->partial, g->digits, g->bucket_box};
    for (void* p : ptrs)
        if (p) (void)hipFree(p);
    delete g;
    return IMBA_OK;
}

int imba_hashgrid_build(ImbaHashGrid* g, const void* photons, int stride, int pos_offset, int count, float radius,
                        void* stream) {
    IMBA_CHECK_ARG(g, "grid is NULL");
    IMBA_CHECK_ARG(count >= 0 && count <= kGridMaxPhotons, "count out of range");
    IMBA_CHECK_ARG(count == 0 || photons, "photons is NULL");
    IMBA_CHECK_ARG(stride >= 12 && stride % 4 == 0 && pos_offset >= 0 && pos_offset % 4 == 0 && pos_offset + 12 <= stride,
                   "stride/pos_offset must be multiples of 4 with the position inside the record");
    IMBA_CHECK_ARG(radius > 0.0f, "radius must be positive");
    bool sync;
    hipStream_t s = resolve_stream(stream, &sync);
    const int table = grid_table_size(g->table_size, count);
    const int reserved = reserve(g, count, table);
    if (reserved) {
        if (g->table_cap == 0 || g->cap < g->count) {  // the last build's buffers are gone
            g->table_size = 0;
            g->count = 0;
        }
        return reserved;
    }
    g->table_size = table;
    g->count = count;
    const unsigned char* ph = (const unsigned char*)photons;
    const int nparts = std::min(kBoundsBlocks, std::max(1, ceil_div(count, kBlock)));
    const int n_tiles = radix_tiles<kSortItems>(count);
    hipLaunchKernelGGL(k_bounds, dim3(nparts), dim3(kBlock), 0, s, ph, stride, pos_offset, count, g->partial);
    hipLaunchKernelGGL(k_grid_keys, dim3(std::max(1, n_tiles)), dim3(kBlock), 0, s, ph, stride, pos_offset, count,
                       g->partial, nparts, g->d_params, radius, table, g->keys_a, n_tiles, g->digits);
    int* keys_sorted = nullptr;
    uint32_t* heads = nullptr;
    if (count > 0) {
        int bits = 1;
        while (bits < 31 && (1 << bits) < table) bits++;  // buckets are < table
        radix_sort<kSortItems>(g->keys_a, g->keys_b, g->vals_a, g->vals_b, count, bits, g->digits, g->order,
                               &keys_sorted, s);
        // The sort's other key buffer: 6 words per 64 slots after the first 64.
        heads = (uint32_t*)(keys_sorted == g->keys_a ? g->keys_b : g->keys_a);
        hipLaunchKernelGGL(k_slots, dim3(ceil_div(count, kBlock * kSlotItems)), dim3(kBlock), 0, s, ph, stride,
                           pos_offset, count, g->order, keys_sorted, g->pos4, g->bucket_box, heads);
    }
    if (table > 0)
        hipLaunchKernelGGL(k_ends, dim3(ceil_div(table, kScanTile)), dim3(kBlock), 0, s, g->cell_ends, table,
                           keys_sorted, count, heads, g->bucket_box);
    IMBA_HIP_TRY(hipGetLastError());
    if (sync) IMBA_HIP_TRY(hipStreamSynchronize(s));
    return IMBA_OK;
}

int imba_hashgrid_query(const ImbaHashGrid* g, const void* queries, int query_stride, int query_offset, int nq, int k,
                        int* out_idx, float* out_dist, int* out_count, void* stream) {
    IMBA_CHECK_ARG(g, "grid is NULL");
    if (k < 1 || k > kQueryMaxK) return fail(IMBA_ERR_INVALID_ARG, "k must be in [1, %d]", kQueryMaxK);
    IMBA_CHECK_ARG(nq >= 0, "nq < 0");
    IMBA_CHECK_ARG(query_stride >= 12 && query_stride % 4 == 0 && query_offset >= 0 && query_offset % 4 == 0 &&
                       query_offset + 12 <= query_stride,
                   "query stride/offset must be multiples of 4 with the position inside the record");
    if (nq == 0) return IMBA_OK;
    IMBA_CHECK_ARG(queries && out_idx && out_count, "NULL buffer");
    if (g->table_size == 0) return fail(IMBA_ERR_INVALID_ARG, "grid has not been built");
    bool sync;
    hipStream_t s = resolve_stream(stream, &sync);
    const unsigned char* qs = (const unsigned char*)queries;
    if (k <= 64) {
        const DeviceProps* p = device_props();
        if (!p) return fail(IMBA_ERR_NO_DEVICE, "no HIP device");
        const int per = queries_per_wave(nq, p->cu_count);
        hipLaunchKernelGGL(k_query_wave, dim3(ceil_div(ceil_div(nq, per), kBlock / 64)), dim3(kBlock), 0, s,
                           g->d_params, g->cell_ends, g->pos4, g->bucket_box, qs, query_stride, query_offset, nq, per,
                           k, out_idx, out_dist, out_count);
    } else
        hipLaunchKernelGGL(k_query_lds, dim3(nq), dim3(64), (size_t)k * 8, s, g->d_params, g->cell_ends, g->pos4, qs,
                           query_stride, query_offset, nq, k, out_idx, out_dist, out_count);
    IMBA_HIP_TRY(hipGetLastError());
    if (sync) IMBA_HIP_TRY(hipStreamSynchronize(s));
    return IMBA_OK;
}

int imba_hashgrid_reset(ImbaHashGrid* g) {
    IMBA_CHECK_ARG(g, "grid is NULL");
    g->table_size = 0;
    g->count = 0;
    return IMBA_OK;
}

int imba_hashgrid_info(const ImbaHashGrid* g, ImbaHashGridInfo* info) {
    IMBA_CHECK_ARG(g && info, "NULL argument");
    GridParams p{};
    IMBA_HIP_TRY(hipMemcpy(&p, g->d_params, sizeof(p), hipMemcpyDeviceToHost));
    info->photon_count = g->count;
    info->table_size = g->table_size;
    for (int k = 0; k < 3; k++) {
        info->bbox_min[k] = p.bmin[k];
        info->bbox_max[k] = p.bmax[k];
    }
    info->radius = p.radius;
    info->radius_sqr = p.radius_sqr;
    info->cell_size = p.cell_size;
    info->inv_cell_size = p.inv_cell_size;
    info->cell_ends = g->cell_ends;
    info->order = g->order;
    info->positions = (const float*)g->pos4;
    return IMBA_OK;
}

__global__ void k_gather_records(const unsigned char* src, int stride, int n, const int* order, unsigned char* dst) {
    const int s = blockIdx.x * 256 + threadIdx.x;
    if (s >= n) return;
    const int i = order[s];
    const int* a = reinterpret_cast<const int*>(src + (size_t)i * stride);
    int* b = reinterpret_cast<int*>(dst + (size_t)s * stride);
    for (int k = 0; k < stride / 4; k++) b[k] = a[k];
}

int imba_hashgrid_gather(const ImbaHashGrid* g, const void* src, int stride, void* dst, void* stream) {
    IMBA_CHECK_ARG(g && src && dst, "NULL argument");
    IMBA_CHECK_ARG(stride > 0 && stride % 4 == 0, "stride must be a positive multiple of 4");
    if (g->count == 0) return IMBA_OK;
    bool sync;
    hipStream_t s = resolve_stream(stream, &sync);
    hipLaunchKernelGGL(k_gather_records, dim3(ceil_div(g->count, 256)), dim3(256), 0, s, (const unsigned char*)src,
                       stride, g->count, g->order, (unsigned char*)dst);
    IMBA_HIP_TRY(hipGetLastError());
    if (sync) IMBA_HIP_TRY(hipStreamSynchronize(s));
    return IMBA_OK;
}

}  // extern "C"
