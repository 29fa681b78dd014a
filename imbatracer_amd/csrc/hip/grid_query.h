// Photon hash grid: parameters, device-side state and the wave's query scan shared by
// the index query (hashgrid.hip, HashGrid::query of rangesearch/rangesearch.h:79-129) and the
// fused vertex-merging launch (vcm.hip).
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

namespace imba {

struct GridParams {
    float bmin[3], bmax[3];
    float radius, radius_sqr, cell_size, inv_cell_size;
    int table_size;
    int count;
};

}  // namespace imba

struct ImbaHashGrid {
    int device = 0;
    int table_size = 0;  // grows only (until imba_hashgrid_reset)
    int table_cap = 0;   // buckets allocated
    int count = 0;
    int cap = 0;         // photon capacity of the per-photon arrays
    int* cell_ends = nullptr;
    int* order = nullptr;
    int* keys_a = nullptr;     // sort buffers (photon_count entries each)
    int* vals_a = nullptr;
    int* keys_b = nullptr;
    int* vals_b = nullptr;
    float4* pos4 = nullptr;    // positions in slot order: x, y, z, photon index bits
    uint32_t* bucket_box = nullptr;  // per bucket: bounds of its photons (lo xyz, hi xyz) as
                                     // ordered_bits, written for the non-empty buckets of the last
                                     // build
    imba::GridParams* d_params = nullptr;
    float* partial = nullptr;  // 6 per bounds block
    int* digits = nullptr;     // the sort's tile counts
    size_t digits_cap = 0;
};

namespace imba {

// The hash of rangesearch/rangesearch.h:136-139 (three primes, xor, modulo the table size).
__device__ __forceinline__ int bucket_of(uint32_t x, uint32_t y, uint32_t z, int table) {
    return (int)(((x * 73856093u) ^ (y * 19349663u) ^ (z * 83492791u)) % (uint32_t)table);
}

constexpr int kDppWaveShr1 = 0x138;  // DPP control: lane i reads lane i - 1 of the wave

// A float's bits mapped to an unsigned integer of the same order (negative floats reversed
// below the positive ones), so that integer min / max are float min / max; and back.
__device__ __forceinline__ uint32_t ordered_bits(float f) {
    const uint32_t u = __float_as_uint(f);
    return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}
__device__ __forceinline__ float from_ordered_bits(uint32_t e) {
    return __uint_as_float((e & 0x80000000u) ? (e & 0x7FFFFFFFu) : ~e);
}

// Squared distance from (qx, qy, qz) to the box of a bucket's photons: a lower bound of every
// photon's squared distance as the scan computes it (float subtraction, squaring and addition
// are monotonic, so a photon inside the box is no nearer than the box).  Only meaningful for a
// bucket that holds photons.
__device__ __forceinline__ float box_dist2(const uint32_t* box, int b, float qx, float qy, float qz) {
    const uint2* e = reinterpret_cast<const uint2*>(box + 6 * (size_t)b);
    const uint2 e0 = e[0], e1 = e[1], e2 = e[2];
    const float lox = from_ordered_bits(e0.x), loy = from_ordered_bits(e0.y), loz = from_ordered_bits(e1.x);
    const float hix = from_ordered_bits(e1.y), hiy = from_ordered_bits(e2.x), hiz = from_ordered_bits(e2.y);
    const float gx = fmaxf(fmaxf(lox - qx, qx - hix), 0.0f);
    const float gy = fmaxf(fmaxf(loy - qy, qy - hiy), 0.0f);
    const float gz = fmaxf(fmaxf(loz - qz, qz - hiz), 0.0f);
    return gx * gx + gy * gy + gz * gz;
}

// The value lane `lane` holds (wave-uniform).
__device__ __forceinline__ float lane_value(float v, int lane) {
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), lane));
}

// The probes of a query: lane 8 q + j holds probe j's bucket range and the squared distance to its
// photons' box for the q-th of the wave's queries.
struct GridProbes {
    int begin, size;
    float lb;
};

// (qx, qy, qz): the position of the lane's query; `active`: it has one.  A query outside the grid
// has eight empty ranges.  All loads of a lane are independent of each other, and those of eight
// queries are in flight together.
__device__ __forceinline__ GridProbes grid_probes(const GridParams& g, const int* ends, const uint32_t* box, float qx,
                                                  float qy, float qz, bool active) {
    GridProbes r{0, 0, 0.0f};
    const bool inside = qx >= g.bmin[0] && qy >= g.bmin[1] && qz >= g.bmin[2] &&
                        qx <= g.bmax[0] && qy <= g.bmax[1] && qz <= g.bmax[2];
    if (!(active && inside && g.count > 0)) return r;
    const int probe = (int)(threadIdx.x & 7);
    const float cx = g.inv_cell_size * (qx - g.bmin[0]);
    const float cy = g.inv_cell_size * (qy - g.bmin[1]);
    const float cz = g.inv_cell_size * (qz - g.bmin[2]);
    const float fx = floorf(cx), fy = floorf(cy), fz = floorf(cz);
    const int x = (int)fx + ((probe & 4) ? ((cx - fx) < 0.5f ? -1 : 1) : 0);
    const int y = (int)fy + ((probe & 2) ? ((cy - fy) < 0.5f ? -1 : 1) : 0);
    const int z = (int)fz + ((probe & 1) ? ((cz - fz) < 0.5f ? -1 : 1) : 0);
    const int b = bucket_of((uint32_t)x, (uint32_t)y, (uint32_t)z, g.table_size);
    r.lb = box_dist2(box, b, qx, qy, qz);  // (an empty bucket's entry holds anything: not used)
    r.begin = ends[b > 0 ? b - 1 : 0];
    r.begin = b > 0 ? r.begin : 0;
    r.size = ends[b] - r.begin;
    return r;
}

// Queries per wave: they share the wave's probing (the hash, the table reads and their latency),
// as long as every SIMD still gets its waves.  600,000 queries, k = 10 / 200,000 queries, k = 64, with
// 1, 2, 4, 8 per wave: 838, 801, 798, 880 us / 632, 636, 679, 850 us.
constexpr int kQueriesPerWave = 2;
inline int queries_per_wave(int nq, int cu_count) {
    int per = kQueriesPerWave;
    while (per > 1 && nq < per * cu_count * 4 * 8) per >>= 1;
    return per;
}

// One query by a whole wave, its probes in lanes `first`..`first` + 7.  The eight probed buckets are
// visited in the reference's order, each bucket's photons scanned in groups of four chunks of 64
// (lane l takes photon base + l of a chunk, so loads are contiguous across the wave and a group's
// are in flight together).
// Candidates within the limit are then inserted one at a time in visiting order with the
// reference's rule; the list itself lives in lanes 0..k-1 (squared distance and id per lane), so
// any k up to 64 fits.  The limit is the radius, or the current k-th distance once the list is
// full, or, where a group holds many candidates, a bound that at least k of the list's entries
// and the group's per-lane minima do not exceed, found by halving.  A candidate beyond any of them
// is beyond the final k-th distance: such a candidate never stays in the list and never
// moves one that does (an insertion only looks at the entries up to it), so the results are those
// of the one-at-a-time scan, equal distances included.  For the same reason a bucket whose photon
// box lies beyond the limit when its turn comes is skipped whole.  The id is the photon index, or
// with SLOTS the photon's slot in the grid order (pos4[slot]).  Returns the list length
// (wave-uniform); lanes >= count hold (0, -1).  Every lane of the wave must call it.
//
// Bound by instruction issue: 690 vector and 500 scalar instructions per query at k = 10 over 1,000
// probed photons, vector issue 95% of the SIMDs' time.  Before the bound (which leaves 11-15 insertions
// of 45), 600,000 queries over 2M photons took 1,557 us, now 785; 200,000 with k = 64 860, now 636;
// with k = 1 265, now 137.  Groups of 2 or 8 chunks and testing a bucket's end per chunk were slower.
template <bool SLOTS>
__device__ __forceinline__ int query_wave_list(const GridParams& g, const float4* pos4, const GridProbes& probes,
                                               int first, float qx, float qy, float qz, int k, float& my_dist,
                                               int& my_id) {
    constexpr int kGroup = 4;    // chunks of 64 photons in flight
    constexpr int kMany = 10;    // candidates of a group above which the bound is worth finding
    constexpr int kHalvings = 7;
    constexpr uint32_t kOctaves = 6;  // the bound is sought down to limit / 64
    // Lanes past a bucket's end and past the list's end hold NaN, which is at most no limit: infinity
    // would be at most an infinite one (an unlimited radius).
    const float none = __int_as_float(0x7fc00000);
    const int lane = (int)(threadIdx.x & 63);
    my_id = -1;
    int count = 0;
    // Distances are compared as their bits where they are wave-uniform (squares' sums are never
    // negative, so the order is the same), which keeps that work on the scalar unit.
    const uint32_t radius_bits = __float_as_uint(g.radius_sqr);
    uint32_t kth = 0x7fc00000u;  // dist[k - 1]; above every distance until the list is full
    my_dist = none;
    for (int j = 0; j < 8; j++) {
        const int beg = __builtin_amdgcn_readlane(probes.begin, first + j);
        const int n = __builtin_amdgcn_readlane(probes.size, first + j);
        const float lbj = lane_value(probes.lb, first + j);
        if (n == 0 || __float_as_uint(lbj) > min(kth, radius_bits)) continue;
        for (int base = 0; base < n; base += 64 * kGroup) {
            float4 p[kGroup];
#pragma unroll
            for (int i = 0; i < kGroup; i++) {
                p[i] = make_float4(none, 0.0f, 0.0f, 0.0f);
                if (base + 64 * i < n && base + 64 * i + lane < n) p[i] = pos4[beg + base + 64 * i + lane];
            }
            float d2[kGroup];
            unsigned long long m[kGroup];
            uint32_t lim = min(kth, radius_bits);
            int candidates = 0;
#pragma unroll
            for (int i = 0; i < kGroup; i++) {
                const float dx = qx - p[i].x, dy = qy - p[i].y, dz = qz - p[i].z;
                d2[i] = dx * dx + dy * dy + dz * dz;
                m[i] = __ballot(d2[i] <= __uint_as_float(lim));
                candidates += __popcll(m[i]);
            }
            if (candidates > kMany) {
                float least = d2[0];
#pragma unroll
                for (int i = 1; i < kGroup; i++) least = fminf(least, d2[i]);
                const float listed = lane < k ? my_dist : none;
                if (__popcll(__ballot(least <= __uint_as_float(lim))) + count >= k) {
                    // lim: always a distance that at least k values do not exceed
                    uint32_t lo = max(lim, kOctaves << 23) - (kOctaves << 23);
                    for (int h = 0; h < kHalvings; h++) {
                        const uint32_t mid = (lo + lim) >> 1;
                        const float f = __uint_as_float(mid);
                        const bool enough = __popcll(__ballot(least <= f)) + __popcll(__ballot(listed <= f)) >= k;
                        lo = enough ? lo : mid;
                        lim = enough ? mid : lim;
                    }
#pragma unroll
                    for (int i = 0; i < kGroup; i++) m[i] = __ballot(d2[i] <= __uint_as_float(lim));
                }
            }
#pragma unroll
            for (int i = 0; i < kGroup; i++) {
                while (m[i]) {
                    const int src = __builtin_ctzll(m[i]);
                    m[i] &= m[i] - 1;
                    const uint32_t dd = (uint32_t)__builtin_amdgcn_readlane(__float_as_int(d2[i]), src);
                    const int id = SLOTS ? beg + base + 64 * i + src
                                         : __builtin_amdgcn_readlane(__float_as_int(p[i].w), src);
                    if (kth < dd) continue;
                    // dd goes after every entry <= dd, but into the last place at the latest (the
                    // reference drops the last entry of a full list first); lanes from k on hold
                    // what was dropped, nothing nearer than the k-th
                    const int pos = min((int)__popcll(__ballot(my_dist <= __uint_as_float(dd))), k - 1);
                    int my_bits = __float_as_int(my_dist);
                    if (lane >= pos) {  // the entries one lane down (wave shift right by one lane, DPP)
                        my_bits = __builtin_amdgcn_update_dpp(my_bits, my_bits, kDppWaveShr1, 0xF, 0xF, false);
                        my_id = __builtin_amdgcn_update_dpp(my_id, my_id, kDppWaveShr1, 0xF, 0xF, false);
                    }
                    my_bits = lane == pos ? (int)dd : my_bits;
                    my_id = lane == pos ? id : my_id;
                    my_dist = __int_as_float(my_bits);
                    count = min(count + 1, k);
                    kth = (uint32_t)__builtin_amdgcn_readlane(my_bits, k - 1);
                }
            }
        }
    }
    if (lane >= count) {
        my_dist = 0.0f;
        my_id = -1;
    }
    return count;
}

}  // namespace imba
