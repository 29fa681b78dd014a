// Stable LSD radix sort of int keys by 8-bit digits, with the entries' original indices as values,
// shared by the material sort and the hash-grid build.
//
// One pass over a digit, in tiles of 256 x ITEMS entries:
//   1. the tile's 256-bin histogram (LDS atomics, one histogram per wave), stored digit-major;
//      the first pass's is left by the kernel that writes the keys (RadixTile);
//   2. k_radix_rows: one block per digit turns its row of tile counts into offsets, the digit's
//      total beside them;
//   3. k_radix_scatter: each wave takes 64 x ITEMS consecutive entries, all loaded at once, and ranks
//      them (eight ballots per 64, one per digit bit, a running count per digit in LDS that only
//      this wave touches, so without barriers); the tile is put in digit order in LDS and
//      written out in that order, neighbouring lanes to neighbouring places.
// Entries with equal digits keep their order, so after the passes over all key bits the entries
// are ordered by key and, for equal keys, by index.
// Traffic per entry and pass: key read twice, value once, both written once (20 B; the first pass
// reads neither values nor, for its counts, keys).  4M entries, 23-bit keys: a pass took 77 us in
// five launches (49 of them the scatter, with four barriers per 256 entries and every lane writing
// where its entry goes), now 38 in three: counts 12, rows 5, scatter 21 (64 MB, 3 TB/s; the ballots
// and LDS work of a tile keep it from the copy rate).
#pragma once

#include <hip/hip_runtime.h>

#include <utility>

namespace imba {
namespace {

constexpr int kRadixBlock = 256;
constexpr int kRadixWaves = kRadixBlock / 64;

template <int ITEMS>
inline int radix_tiles(int n) {
    return (n + kRadixBlock * ITEMS - 1) / (kRadixBlock * ITEMS);
}

// A block's tile: its histogram of one digit.  Entry `it` of a thread is index(it).
template <int ITEMS>
struct RadixTile {
    int hist[kRadixWaves][256];

    __device__ __forceinline__ static int index(int it) {
        return (int)blockIdx.x * kRadixBlock * ITEMS + it * kRadixBlock + (int)threadIdx.x;
    }
    __device__ __forceinline__ void clear() {
#pragma unroll
        for (int w = 0; w < kRadixWaves; w++) hist[w][threadIdx.x] = 0;
        __syncthreads();
    }
    __device__ __forceinline__ void add(int digit) { atomicAdd(&hist[threadIdx.x >> 6][digit], 1); }
    // The tile's counts to counts[digit][tile].
    __device__ __forceinline__ void store(int* counts, int n_tiles) {
        __syncthreads();
        int c = 0;
#pragma unroll
        for (int w = 0; w < kRadixWaves; w++) c += hist[w][threadIdx.x];
        counts[(size_t)threadIdx.x * n_tiles + blockIdx.x] = c;
    }
};

template <int ITEMS>
__global__ __launch_bounds__(kRadixBlock) void k_radix_hist(const int* __restrict__ keys, int n, int shift,
                                                            int n_tiles, int* counts) {
    __shared__ RadixTile<ITEMS> tile;
    tile.clear();
    int key[ITEMS];
#pragma unroll
    for (int it = 0; it < ITEMS; it++) key[it] = tile.index(it) < n ? keys[tile.index(it)] : 0;
#pragma unroll
    for (int it = 0; it < ITEMS; it++)
        if (tile.index(it) < n) tile.add((key[it] >> shift) & 255);
    tile.store(counts, n_tiles);
}

// Inclusive sum over the block's threads; `ws` holds an int per wave.
__device__ __forceinline__ int radix_block_scan(int v, int* ws) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    for (int o = 1; o < 64; o <<= 1) {
        const int y = __shfl_up(v, o, 64);
        if (lane >= o) v += y;
    }
    if (lane == 63) ws[wave] = v;
    __syncthreads();
    for (int w = 0; w < wave; w++) v += ws[w];
    __syncthreads();
    return v;
}

// Block d: exclusive scan of row d of the counts in place, its sum to totals[d].
__global__ __launch_bounds__(kRadixBlock) void k_radix_rows(int* counts, int n_tiles, int* totals) {
    __shared__ int ws[kRadixWaves];
    __shared__ int last;
    int* row = counts + (size_t)blockIdx.x * n_tiles;
    int run = 0;
    for (int base = 0; base < n_tiles; base += kRadixBlock) {
        const int i = base + (int)threadIdx.x;
        const int c = i < n_tiles ? row[i] : 0;
        const int x = radix_block_scan(c, ws);
        if (i < n_tiles) row[i] = run + x - c;
        if (threadIdx.x == kRadixBlock - 1) last = x;
        __syncthreads();
        run += last;
    }
    if (threadIdx.x == 0) totals[blockIdx.x] = run;
}

// FIRST: the values are the entries' indices (vals_in is not read).
template <int ITEMS, bool FIRST>
__global__ __launch_bounds__(kRadixBlock) void k_radix_scatter(const int* __restrict__ keys_in,
                                                               const int* __restrict__ vals_in, int n, int shift,
                                                               int n_tiles, const int* __restrict__ offsets,
                                                               const int* __restrict__ totals, int* keys_out,
                                                               int* vals_out) {
    constexpr int kTile = kRadixBlock * ITEMS;
    __shared__ int count[kRadixWaves][256];  // a wave's entries per digit, then the waves' before it
    __shared__ int start[256];               // the digit's first place in the tile
    __shared__ int move[256];                // what takes a place in the tile to one in the output
    __shared__ int ws[kRadixWaves];
    __shared__ int skey[kTile], sval[kTile];
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    const unsigned long long lt = lane ? (~0ull >> (64 - lane)) : 0ull;  // lanes below this one
    const int base = blockIdx.x * kTile;
    const int first = base + wave * 64 * ITEMS + lane;
    int key[ITEMS], val[ITEMS], rank[ITEMS];
#pragma unroll
    for (int it = 0; it < ITEMS; it++) {
        const int i = first + it * 64;
        key[it] = i < n ? keys_in[i] : 0;
        val[it] = FIRST ? i : i < n ? vals_in[i] : 0;
    }
    const int digit_total = totals[t], tile_offset = offsets[(size_t)t * n_tiles + blockIdx.x];
    for (int k = lane; k < 256; k += 64) count[wave][k] = 0;
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (int it = 0; it < ITEMS; it++) {
        const bool valid = first + it * 64 < n;
        const int digit = (key[it] >> shift) & 255;
        unsigned long long same = __ballot(valid);  // lanes with the same digit
#pragma unroll
        for (int b = 0; b < 8; b++) {
            const unsigned long long bits = __ballot((digit >> b) & 1);
            same &= ((digit >> b) & 1) ? bits : ~bits;
        }
        const int before = __popcll(same & lt);
        rank[it] = count[wave][digit] + before;  // every lane reads before the first of them adds
        __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
        __builtin_amdgcn_wave_barrier();
        if (valid && before == 0) count[wave][digit] = rank[it] + __popcll(same);
        __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
        __builtin_amdgcn_wave_barrier();
    }
    __syncthreads();
    int tile_total = 0;
#pragma unroll
    for (int w = 0; w < kRadixWaves; w++) {
        const int c = count[w][t];
        count[w][t] = tile_total;
        tile_total += c;
    }
    const int tile_start = radix_block_scan(tile_total, ws) - tile_total;
    const int digit_start = radix_block_scan(digit_total, ws) - digit_total;
    start[t] = tile_start;
    move[t] = digit_start + tile_offset - tile_start;
    __syncthreads();
#pragma unroll
    for (int it = 0; it < ITEMS; it++) {
        if (first + it * 64 < n) {
            const int digit = (key[it] >> shift) & 255;
            const int at = start[digit] + count[wave][digit] + rank[it];
            skey[at] = key[it];
            sval[at] = val[it];
        }
    }
    __syncthreads();
    const int left = min(kTile, n - base);
#pragma unroll
    for (int it = 0; it < ITEMS; it++) {
        const int i = it * kRadixBlock + t;
        if (i < left) {
            const int k = skey[i];
            const int to = move[(k >> shift) & 255] + i;
            keys_out[to] = k;
            vals_out[to] = sval[i];
        }
    }
}

// Ints of the `counts` workspace radix_sort needs for n entries: the tile counts, then the digits'
// totals.
template <int ITEMS>
inline size_t radix_counts_size(int n) {
    return (size_t)256 * radix_tiles<ITEMS>(n) + 256;
}

// Sorts n keys (in [0, 2^bits)) from keys_a using keys_b as the other buffer; vals_a and vals_b
// hold n ints each for the values of the passes between.  `counts` holds radix_counts_size<ITEMS>(n)
// ints, the first 256 x tiles of them the tile counts of the lowest digit (RadixTile).  The last
// pass writes the indices to vals_final; *keys_sorted is set to the buffer holding the sorted
// keys.  Launch errors are left for the caller's hipGetLastError.
template <int ITEMS>
void radix_sort(int* keys_a, int* keys_b, int* vals_a, int* vals_b, int n, int bits, int* counts, int* vals_final,
                int** keys_sorted, hipStream_t s) {
    const int passes = bits <= 8 ? 1 : (bits + 7) / 8;
    const int n_tiles = radix_tiles<ITEMS>(n);
    int* totals = counts + (size_t)256 * n_tiles;
    for (int p = 0; p < passes; p++) {
        const int shift = 8 * p;
        int* vo = p == passes - 1 ? vals_final : vals_b;
        if (p > 0)
            hipLaunchKernelGGL(k_radix_hist<ITEMS>, dim3(n_tiles), dim3(kRadixBlock), 0, s, keys_a, n, shift, n_tiles,
                               counts);
        hipLaunchKernelGGL(k_radix_rows, dim3(256), dim3(kRadixBlock), 0, s, counts, n_tiles, totals);
        if (p == 0)
            hipLaunchKernelGGL((k_radix_scatter<ITEMS, true>), dim3(n_tiles), dim3(kRadixBlock), 0, s, keys_a,
                               (const int*)nullptr, n, shift, n_tiles, counts, totals, keys_b, vo);
        else
            hipLaunchKernelGGL((k_radix_scatter<ITEMS, false>), dim3(n_tiles), dim3(kRadixBlock), 0, s, keys_a, vals_a,
                               n, shift, n_tiles, counts, totals, keys_b, vo);
        std::swap(keys_a, keys_b);
        std::swap(vals_a, vals_b);
    }
    *keys_sorted = keys_a;
}

}  // namespace
}  // namespace imba
