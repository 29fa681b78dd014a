// Closest-hit and any-hit traversal of two-level BVH2 scenes on gfx950.
//
// Replaces the AnyDSL kernels intersect_gpu_masked_instanced / occluded_gpu_masked_instanced
// that the reference calls at render/scheduling/ray_queue.h:297-308 and 347-358 (their source
// is not part of the reference).  Layouts are those written by the reference's GPU adapters
// (core/gpu_adapter.cpp): 64-byte BVH2 nodes, three Vec4 per triangle with the triangle id in
// v1.w and the leaf end flagged by the bit pattern 0x80000000 in v2.w, 64-byte instance
// records ending a top-level leaf with pad = {-1,-1}.
//
// Per ray the traversal is depth first: the child boxes of a node are tested, the nearest hit
// child (ties: the lower one) is visited first and the others are pushed.  Entering an instance
// transforms the ray into object space and remembers the stack depth; when the stack falls
// back to that depth the next instance of the same leaf is entered, or the world ray is
// restored.  Arithmetic (fixed, shared with the CPU restatement used as the checker):
//   box:      t = fma(bound, 1/d', -o * (1/d')), d' = d or +-1e-9 when |d| < 1e-9;
//             near = max(max(min x, min y), max(min z, tmin)),
//             far  = min(min(max x, max y), min(max z, t_best)); hit when near <= far
//   triangle: e1 = v0 - v1, e2 = v2 - v0, n = e1 x e2, c = v0 - o, r = d x c,
//             det = n.d, U = r.e2, V = r.e1, T = n.c (cross and dot with fma as below);
//             with signs folded by det: U >= 0, V >= 0, |det| - U - V >= 0, det != 0;
//             t = T / |det|, u = U / |det|
//   cross(a, b) = (fma(a.y, b.z, -(a.z b.y)), fma(a.z, b.x, -(a.x b.z)), fma(a.x, b.y, -(a.y b.x)))
//   dot(a, b)   = fma(a.x, b.x, fma(a.y, b.y, a.z b.z))
//   instance:   o' = M (o, 1), d' = M (d, 0) with row sums fma(m0, x, fma(m1, y, fma(m2, z, m3)))
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

namespace imba {

struct TraceArgs {
    const float4* nodes;  int n_nodes;
    const float4* inst;   int n_inst;
    const float4* tris;   int n_tris4;
    const int4* indices;  int n_tri_ids;     // triangles described by `indices`
    const float2* texcoords; int n_texcoords;
    const int* masks;     int n_masks;       // 3 ints per mask: width, height, offset
    const unsigned char* mask_buf; int mask_buf_size;
    const float4* rays;   int4* hits; int count; int root;
    uint32_t* counts;     // 3 per ray (stats variant), or null
    uint32_t* depth_hist; // stats variant: rays by the deepest stack entry they used (64 bins,
                          // the last one for 63 and deeper), or null
    int* err;             // incremented once per ray that met a malformed structure
    int* spill;           // global stack entries beyond the LDS part
    int spill_depth;      // spill entries per thread
    int spill_stride;     // threads that may spill (the first of the grid)
    int* work_counter;    // persistent variant: next ray to fetch
    const int* count_dev; // device ray count read when the launch runs (<= count), or null
    int quad;             // quantized tree: a launch of at most this many rays gives each ray four lanes
};

// Rays of this launch: count, or the device count clamped to [0, count].
__device__ __forceinline__ int launch_count(const TraceArgs& a) {
    return a.count_dev ? min(max(*a.count_dev, 0), a.count) : a.count;
}

constexpr int kNoNode = INT32_MIN;
constexpr int kDummyChild = 0x76543210;
constexpr uint32_t kLeafEnd = 0x80000000u;

struct RaySpace {
    float ox, oy, oz, dx, dy, dz;
    float idx, idy, idz, oidx, oidy, oidz;
};

__device__ __forceinline__ float safe_dir(float d) { return fabsf(d) < 1e-9f ? copysignf(1e-9f, d) : d; }

__device__ __forceinline__ void setup_space(RaySpace& r) {
    r.idx = 1.0f / safe_dir(r.dx);
    r.idy = 1.0f / safe_dir(r.dy);
    r.idz = 1.0f / safe_dir(r.dz);
    r.oidx = r.ox * r.idx;
    r.oidy = r.oy * r.idy;
    r.oidz = r.oz * r.idz;
}

__device__ __forceinline__ bool box_hit(const RaySpace& r, float lx, float hx, float ly, float hy, float lz, float hz,
                                        float tmin, float tmax, float& tnear) {
    const float t0x = fmaf(lx, r.idx, -r.oidx), t1x = fmaf(hx, r.idx, -r.oidx);
    const float t0y = fmaf(ly, r.idy, -r.oidy), t1y = fmaf(hy, r.idy, -r.oidy);
    const float t0z = fmaf(lz, r.idz, -r.oidz), t1z = fmaf(hz, r.idz, -r.oidz);
    tnear = fmaxf(fmaxf(fminf(t0x, t1x), fminf(t0y, t1y)), fmaxf(fminf(t0z, t1z), tmin));
    const float tfar = fminf(fminf(fmaxf(t0x, t1x), fmaxf(t0y, t1y)), fminf(fmaxf(t0z, t1z), tmax));
    return tnear <= tfar;
}

// Returns true when the ray meets the triangle (edges included, det != 0); t, u, v are
// then the distance and the barycentric weights of v1 and v2.
__device__ __forceinline__ bool tri_hit(const RaySpace& r, const float4& a, const float4& b, const float4& c,
                                        float& t, float& u, float& v) {
    const float e1x = a.x - b.x, e1y = a.y - b.y, e1z = a.z - b.z;
    const float e2x = c.x - a.x, e2y = c.y - a.y, e2z = c.z - a.z;
    const float nx = fmaf(e1y, e2z, -(e1z * e2y));
    const float ny = fmaf(e1z, e2x, -(e1x * e2z));
    const float nz = fmaf(e1x, e2y, -(e1y * e2x));
    const float cx = a.x - r.ox, cy = a.y - r.oy, cz = a.z - r.oz;
    const float rx = fmaf(r.dy, cz, -(r.dz * cy));
    const float ry = fmaf(r.dz, cx, -(r.dx * cz));
    const float rz = fmaf(r.dx, cy, -(r.dy * cx));
    const float det = fmaf(nx, r.dx, fmaf(ny, r.dy, nz * r.dz));
    const float U = fmaf(rx, e2x, fmaf(ry, e2y, rz * e2z));
    const float V = fmaf(rx, e1x, fmaf(ry, e1y, rz * e1z));
    const float T = fmaf(nx, cx, fmaf(ny, cy, nz * cz));
    const bool neg = det < 0.0f;
    const float ad = fabsf(det);
    const float us = neg ? -U : U;
    const float vs = neg ? -V : V;
    const float w = (ad - us) - vs;
    if (!(us >= 0.0f && vs >= 0.0f && w >= 0.0f && det != 0.0f)) return false;
    const float ts = neg ? -T : T;
    t = ts / ad;
    u = us / ad;
    v = vs / ad;
    return true;
}

// Opacity of the material mask at the hit (texel: wrap the interpolated texcoords to [0,1),
// scale by the mask size, truncate, clamp to the last texel).  Returns 1 when opaque, 0 when
// transparent, and 3 (opaque, bit 1 set) when the scene arrays are inconsistent.
__device__ __forceinline__ int texel_opaque(const TraceArgs& a, int tri, float u, float v) {
    if ((unsigned)tri >= (unsigned)a.n_tri_ids) return 3;
    const int4 ind = a.indices[tri];
    if ((unsigned)ind.w >= (unsigned)a.n_masks) return 3;
    const int w = a.masks[3 * ind.w + 0], h = a.masks[3 * ind.w + 1], off = a.masks[3 * ind.w + 2];
    int texel = 0;
    if (!(w == 1 && h == 1)) {
        if ((unsigned)ind.x >= (unsigned)a.n_texcoords || (unsigned)ind.y >= (unsigned)a.n_texcoords ||
            (unsigned)ind.z >= (unsigned)a.n_texcoords)
            return 3;
        const float2 t0 = a.texcoords[ind.x], t1 = a.texcoords[ind.y], t2 = a.texcoords[ind.z];
        const float w0 = (1.0f - u) - v;
        const float s = fmaf(t0.x, w0, fmaf(t1.x, u, t2.x * v));
        const float q = fmaf(t0.y, w0, fmaf(t1.y, u, t2.y * v));
        const float fs = (s - floorf(s)) * (float)w;
        const float fq = (q - floorf(q)) * (float)h;
        const int xi = (fs >= 0.0f && fs < (float)w) ? (int)fs : (fs >= (float)w ? w - 1 : 0);
        const int yi = (fq >= 0.0f && fq < (float)h) ? (int)fq : (fq >= (float)h ? h - 1 : 0);
        texel = yi * w + xi;
    }
    const long long at = (long long)off + texel;
    if (at < 0 || at >= a.mask_buf_size) return 3;
    return a.mask_buf[at] != 0 ? 1 : 0;
}

// Address-space qualifiers for the device pass (the host pass sees plain pointers).
#if defined(__HIP_DEVICE_COMPILE__)
#define IMBA_AS(n) __attribute__((address_space(n)))
#else
#define IMBA_AS(n)
#endif

// The LDS (address space 3) view of a pointer into a kernel's __shared__ memory: accesses through
// it are ds_read / ds_write, not flat accesses (which the compiler otherwise emits when an LDS
// and a global access are merged into one load through a selected pointer).
template <typename T>
__device__ __forceinline__ IMBA_AS(3) T* lds_view(T* p) {
    return (IMBA_AS(3) T*)p;
}

// The global (address space 1) view of a scene or queue array: loads through it are
// global_load, not flat_load, also where the pointer itself was read from memory (the batched
// kernel's queue table), which the compiler cannot otherwise place.
template <typename T>
__device__ __forceinline__ const IMBA_AS(1) T* gview(const T* p) {
    return (const IMBA_AS(1) T*)p;
}
template <typename T>
__device__ __forceinline__ IMBA_AS(1) T* gview_w(T* p) {
    return (IMBA_AS(1) T*)p;
}

// Per-lane traversal stack: entry 0..sp-1 in LDS ([depth][lane], conflict free), then in the
// global spill buffer.  (Holding the top entry in a register measured no faster.)
template <int BLOCK, int STACK_LDS>
struct LaneStack {
    int* lds;     // [STACK_LDS][BLOCK]
    int* spill;   // [spill_depth][threads] or null
    int spill_depth;
    int lane_slot;   // threadIdx.x
    int spill_slot;  // global thread index
    int spill_stride;
    int sp;

    __device__ __forceinline__ bool push(int v) {
        // (the capacity test only on the spill path: testing it first for every push measured
        // 14% slower on the deep trees of 256 queues over 10K-4M random triangles)
        if (sp < STACK_LDS) {
            lds_view(lds)[sp * BLOCK + lane_slot] = v;
        } else {
            const int k = sp - STACK_LDS;
            if (k >= spill_depth) return false;
            spill[(size_t)k * spill_stride + spill_slot] = v;
        }
        sp++;
        return true;
    }
    // Pushes the first n of c1, c2, c3 (n <= 3), the last one deepest.
    __device__ __forceinline__ bool push3(int c1, int c2, int c3, int n) {
        if (sp + 3 <= STACK_LDS) {
            // written without branches: an entry past the new top is overwritten by a later push
            auto* p = lds_view(lds) + sp * BLOCK + lane_slot;
            p[0] = n >= 3 ? c3 : n == 2 ? c2 : c1;
            p[BLOCK] = n >= 3 ? c2 : c1;
            p[2 * BLOCK] = c1;
            sp += n;
            return true;
        }
        bool ok = true;
        if (n >= 3) ok &= push(c3);
        if (n >= 2) ok &= push(c2);
        if (n >= 1) ok &= push(c1);
        return ok;
    }
    __device__ __forceinline__ int pop() {
        sp--;
        if (sp < STACK_LDS) return lds_view(lds)[sp * BLOCK + lane_slot];
        return spill[(size_t)(sp - STACK_LDS) * spill_stride + spill_slot];
    }
    // For a quad working on this stack (advance_quad): whether it can hold `top` entries, and a
    // write of entry e.
    __device__ __forceinline__ bool holds(int top) const { return top <= STACK_LDS || top - STACK_LDS <= spill_depth; }
    __device__ __forceinline__ void put(int e, int v) {
        if (e < STACK_LDS) lds_view(lds)[e * BLOCK + lane_slot] = v;
        else spill[(size_t)(e - STACK_LDS) * spill_stride + spill_slot] = v;
    }
};

// The stack of a ray that has a quad of lanes from the start: the LDS of its four lanes.
template <int BLOCK, int STACK_LDS>
struct QuadStack {
    int* lds;  // [4 * STACK_LDS][BLOCK / 4], the quad's column
    int sp;

    __device__ __forceinline__ int pop() { return lds_view(lds)[--sp * (BLOCK / 4)]; }
    __device__ __forceinline__ bool holds(int top) const { return top <= 4 * STACK_LDS; }
    __device__ __forceinline__ void put(int e, int v) { lds_view(lds)[e * (BLOCK / 4)] = v; }
};

__device__ __forceinline__ float4 as_float4(const uint4& u) {
    return make_float4(__uint_as_float(u.x), __uint_as_float(u.y), __uint_as_float(u.z), __uint_as_float(u.w));
}


// The world-space ray, kept while the ray is inside an instance.
struct WorldRay {
    float ox, oy, oz, dx, dy, dz;
    float idx, idy, idz;  // 1 / safe_dir(d), as setup_space computes them
};

// What a ray does in its next step: a node, a triangle of the current leaf, an instance, or
// (kNone) whatever comes off the stack.
enum : int { kNode = 0, kTri = 1, kInst = 2, kNone = 3 };

// Traversal state of one ray.  Every member is assigned from every path of a step by value: a
// member stored on one side of a branch and another on the other side is merged into one store
// through a selected address, which puts the state into scratch memory.
struct TraceState {
    WorldRay world;  // world-space ray (its reciprocals are recomputed when the ray returns to it)
    RaySpace cs;     // ray in the space of the current level (world or an instance's object space)
    float tmin;      // the ray's tmax is best_t until a hit
    float best_t, best_u;
    int best_tri, best_inst;
    int kind;        // what comes next
    int item;        // its index (node, Vec4 of the triangle's first vertex, instance record)
    int inst_id;     // id of the current instance
    int inst_next;   // the next instance record of the same leaf, -1: none
    int inst_sp;     // stack depth when the instance was entered, -1 in world space
    int bad;         // the ray met a malformed structure
    uint32_t cn, ct, ci;  // visit counts (stats variant)
    uint32_t cd;          // deepest stack entry used (stats variant)
};

// The current space becomes world space (the reciprocals kept from the start: the values
// setup_space gives).
__device__ __forceinline__ void to_world(TraceState& s) {
    s.cs.ox = s.world.ox; s.cs.oy = s.world.oy; s.cs.oz = s.world.oz;
    s.cs.dx = s.world.dx; s.cs.dy = s.world.dy; s.cs.dz = s.world.dz;
    s.cs.idx = s.world.idx; s.cs.idy = s.world.idy; s.cs.idz = s.world.idz;
    s.cs.oidx = s.cs.ox * s.cs.idx;
    s.cs.oidy = s.cs.oy * s.cs.idy;
    s.cs.oidz = s.cs.oz * s.cs.idz;
}

__device__ __forceinline__ void state_init(TraceState& s, const float4& ro, const float4& rd, int root) {
    s.world.ox = ro.x; s.world.oy = ro.y; s.world.oz = ro.z;
    s.world.dx = rd.x; s.world.dy = rd.y; s.world.dz = rd.z;
    s.cs.ox = ro.x; s.cs.oy = ro.y; s.cs.oz = ro.z;
    s.cs.dx = rd.x; s.cs.dy = rd.y; s.cs.dz = rd.z;
    setup_space(s.cs);
    s.world.idx = s.cs.idx; s.world.idy = s.cs.idy; s.world.idz = s.cs.idz;
    s.tmin = ro.w;
    s.best_t = rd.w;
    s.best_u = 0.0f;
    s.best_tri = -1;
    s.best_inst = -1;
    s.kind = kNode;
    s.item = root;
    s.inst_id = -1;
    s.inst_next = -1;
    s.inst_sp = -1;
    s.bad = 0;
    s.cn = s.ct = s.ci = s.cd = 0;
}

// Instance record i (r0..r2 its transform, r3 its id, root and list end): the ray goes to its
// object space and on to the instance's root node.
template <bool STATS>
__device__ __forceinline__ int enter_instance(TraceState& s, const uint4& r0, const uint4& r1, const uint4& r2,
                                               const uint4& r3, int sp) {
    const float4 m0 = as_float4(r0), m1 = as_float4(r1), m2 = as_float4(r2);
    if (STATS) s.ci++;
    const WorldRay& w = s.world;
    s.cs.ox = fmaf(m0.x, w.ox, fmaf(m0.y, w.oy, fmaf(m0.z, w.oz, m0.w)));
    s.cs.oy = fmaf(m1.x, w.ox, fmaf(m1.y, w.oy, fmaf(m1.z, w.oz, m1.w)));
    s.cs.oz = fmaf(m2.x, w.ox, fmaf(m2.y, w.oy, fmaf(m2.z, w.oz, m2.w)));
    s.cs.dx = fmaf(m0.x, w.dx, fmaf(m0.y, w.dy, m0.z * w.dz));
    s.cs.dy = fmaf(m1.x, w.dx, fmaf(m1.y, w.dy, m1.z * w.dz));
    s.cs.dz = fmaf(m2.x, w.dx, fmaf(m2.y, w.dy, m2.z * w.dz));
    if (__float_as_uint(s.cs.dx) == __float_as_uint(w.dx) && __float_as_uint(s.cs.dy) == __float_as_uint(w.dy) &&
        __float_as_uint(s.cs.dz) == __float_as_uint(w.dz)) {
        // the direction is unchanged (a translation or the identity): the world reciprocals
        s.cs.idx = w.idx; s.cs.idy = w.idy; s.cs.idz = w.idz;
        s.cs.oidx = s.cs.ox * s.cs.idx;
        s.cs.oidy = s.cs.oy * s.cs.idy;
        s.cs.oidz = s.cs.oz * s.cs.idz;
    } else {
        setup_space(s.cs);
    }
    s.inst_id = (int)r3.x;
    s.inst_next = (int)r3.z == -1 ? -1 : s.item + 1;
    s.inst_sp = sp;
    return (int)r3.y & 0x7fffffff;  // out of range (a negative root included): the next step's bounds check
}

// One inner node of the BVH2: both child boxes are tested, the nearer hit child (ties: left)
// is next and the other is pushed.
template <int BLOCK, int STACK_LDS, bool STATS>
__device__ __forceinline__ int node_step2(TraceState& s, LaneStack<BLOCK, STACK_LDS>& st, const uint4& r0,
                                           const uint4& r1, const uint4& r2, const uint4& r3) {
    const int n = s.item;
    const float4 n0 = as_float4(r0), n1 = as_float4(r1), n2 = as_float4(r2);
    const int cl = (int)r3.x, cr = (int)r3.y;
    if (STATS) s.cn++;
    float tl = 0.0f, tr = 0.0f;
    bool hl = box_hit(s.cs, n0.x, n0.y, n0.z, n0.w, n1.x, n1.y, s.tmin, s.best_t, tl);
    bool hr = cr != kDummyChild && box_hit(s.cs, n1.z, n1.w, n2.x, n2.y, n2.z, n2.w, s.tmin, s.best_t, tr);
    if (hl && cl >= 0 && cl <= n) { hl = false; s.bad = 1; }
    if (hr && cr >= 0 && cr <= n) { hr = false; s.bad = 1; }
    const bool left_first = hl && !(hr && tr < tl);
    if (hl && hr) {
        if (!st.push(left_first ? cr : cl)) s.bad = 1;
        if (STATS) s.cd = max(s.cd, (uint32_t)st.sp);
    }
    return hl || hr ? (left_first ? cl : cr) : kNoNode;
}

// Ordered exchange of two (distance, link) pairs: the nearer first, the lower slot on a tie.
__device__ __forceinline__ void order2(float& da, int& ca, float& db, int& cb) {
    const bool sw = db < da;
    const float d = sw ? db : da;
    const int c = sw ? cb : ca;
    db = sw ? da : db;
    cb = sw ? ca : cb;
    da = d;
    ca = c;
}

// The hit children of a 4-wide node, given their distances (infinity: not hit): the nearest is
// next, the others are pushed, farthest deepest.
template <int BLOCK, int STACK_LDS, bool STATS>
__device__ __forceinline__ int descend4(TraceState& s, LaneStack<BLOCK, STACK_LDS>& st, float e0, float e1, float e2,
                                         float e3, int c0, int c1, int c2, int c3, int cnt) {
    // sorting network; misses (at infinity) end up last
    order2(e0, c0, e1, c1);
    order2(e2, c2, e3, c3);
    order2(e0, c0, e2, c2);
    order2(e1, c1, e3, c3);
    order2(e1, c1, e2, c2);
    if (!st.push3(c1, c2, c3, max(cnt - 1, 0))) s.bad = 1;
    if (STATS) s.cd = max(s.cd, (uint32_t)st.sp);
    return cnt ? c0 : kNoNode;
}

// One node of the 4-wide tree (ImbaNode4 layout: 8 float4 = min_x, max_x, min_y, max_y, min_z,
// max_z, children, count): the used child boxes are tested.
template <int BLOCK, int STACK_LDS, bool STATS>
__device__ __forceinline__ int node_step4(const TraceArgs& a, TraceState& s, LaneStack<BLOCK, STACK_LDS>& st,
                                           const uint4& r0, const uint4& r1, const uint4& r2, const uint4& r3) {
    const int n = s.item;
    const auto* p = gview(a.nodes + 8 * (size_t)n);
    const float4 lz = p[4], hz = p[5];
    const int4 ch = gview(reinterpret_cast<const int4*>(a.nodes + 8 * (size_t)n))[6];
    const float4 lx = as_float4(r0), hx = as_float4(r1), ly = as_float4(r2), hy = as_float4(r3);
    if (STATS) s.cn++;
    const float inf = __int_as_float(0x7f800000);
    float d[4];
    int cnt = 0;
#pragma unroll
    for (int j = 0; j < 4; j++) {
        auto at = [&](const float4& v) { return j == 0 ? v.x : j == 1 ? v.y : j == 2 ? v.z : v.w; };
        const int c = j == 0 ? ch.x : j == 1 ? ch.y : j == 2 ? ch.z : ch.w;
        // a used link is a leaf (negative) or a node after this one; anything else (0: unused) is
        // not followed
        const bool h = (unsigned)c > (unsigned)n &&
                       box_hit(s.cs, at(lx), at(hx), at(ly), at(hy), at(lz), at(hz), s.tmin, s.best_t, d[j]);
        cnt += h;
        d[j] = h ? d[j] : inf;
    }
    return descend4<BLOCK, STACK_LDS, STATS>(s, st, d[0], d[1], d[2], d[3], ch.x, ch.y, ch.z, ch.w, cnt);
}

// Origin and steps of a quantized 4-wide node's child bounds (its first 16 bytes); a bound is
// fma(byte, 2^e, origin).
struct QuantFrame {
    float ox, oy, oz, sx, sy, sz;
    __device__ __forceinline__ explicit QuantFrame(const uint4& w)
        : ox(__uint_as_float(w.x)), oy(__uint_as_float(w.y)), oz(__uint_as_float(w.z)),
          sx(ldexpf(1.0f, (int)(int8_t)(w.w & 255u))), sy(ldexpf(1.0f, (int)(int8_t)((w.w >> 8) & 255u))),
          sz(ldexpf(1.0f, (int)(int8_t)((w.w >> 16) & 255u))) {}
};
__device__ __forceinline__ float byte_of(uint32_t word, int k) { return (float)((word >> (8 * k)) & 255u); }

// box_hit for the box whose near and far bounds are byte k* of the words n* and f*: t grows with
// the bound when the direction's reciprocal is positive and falls when it is negative (fma rounds
// monotonically), so the bounds chosen by the direction's sign give the min and max of box_hit.
__device__ __forceinline__ bool quant_box_hit(const TraceState& s, const QuantFrame& q, uint32_t nx, int knx,
                                              uint32_t fx, int kfx, uint32_t ny, int kny, uint32_t fy, int kfy,
                                              uint32_t nz, int knz, uint32_t fz, int kfz, float& tnear) {
    const RaySpace& r = s.cs;
    const float t0x = fmaf(fmaf(byte_of(nx, knx), q.sx, q.ox), r.idx, -r.oidx);
    const float t1x = fmaf(fmaf(byte_of(fx, kfx), q.sx, q.ox), r.idx, -r.oidx);
    const float t0y = fmaf(fmaf(byte_of(ny, kny), q.sy, q.oy), r.idy, -r.oidy);
    const float t1y = fmaf(fmaf(byte_of(fy, kfy), q.sy, q.oy), r.idy, -r.oidy);
    const float t0z = fmaf(fmaf(byte_of(nz, knz), q.sz, q.oz), r.idz, -r.oidz);
    const float t1z = fmaf(fmaf(byte_of(fz, kfz), q.sz, q.oz), r.idz, -r.oidz);
    tnear = fmaxf(fmaxf(t0x, t0y), fmaxf(t0z, s.tmin));
    return tnear <= fminf(fminf(t1x, t1y), fminf(t1z, s.best_t));
}

// One node of the quantized 4-wide tree (64 B: origin and exponents, children, 8-bit child
// bounds per axis); otherwise as node_step4.  The dequantized boxes contain the exact ones.
template <int BLOCK, int STACK_LDS, bool STATS>
__device__ __forceinline__ int node_step4q(TraceState& s, LaneStack<BLOCK, STACK_LDS>& st, const uint4& w0,
                                           const uint4& w1, const uint4& w2, const uint4& w3) {
    const uint32_t n = (uint32_t)s.item;
    if (STATS) s.cn++;
    const QuantFrame q(w0);
    const bool px = s.cs.idx >= 0.0f, py = s.cs.idy >= 0.0f, pz = s.cs.idz >= 0.0f;
    const uint32_t nx = px ? w2.x : w2.y, fx = px ? w2.y : w2.x;
    const uint32_t ny = py ? w2.z : w2.w, fy = py ? w2.w : w2.z;
    const uint32_t nz = pz ? w3.x : w3.y, fz = pz ? w3.y : w3.x;
    float d[4];
    int cnt = 0;
#pragma unroll
    for (int j = 0; j < 4; j++) {
        const uint32_t c = j == 0 ? w1.x : j == 1 ? w1.y : j == 2 ? w1.z : w1.w;
        const bool h = quant_box_hit(s, q, nx, j, fx, j, ny, j, fy, j, nz, j, fz, j, d[j]) && c > n;
        cnt += h;
        d[j] = h ? d[j] : __int_as_float(0x7f800000);
    }
    return descend4<BLOCK, STACK_LDS, STATS>(s, st, d[0], d[1], d[2], d[3], (int)w1.x, (int)w1.y, (int)w1.z, (int)w1.w,
                                             cnt);
}

// Whether a hit at t on triangle tid of the current instance replaces the ray's best one.
template <bool ANY>
__device__ __forceinline__ bool is_better(const TraceState& s, float t, int tid) {
    if (ANY) return t <= s.best_t;
    return t < s.best_t || (t == s.best_t && ((unsigned)tid < (unsigned)s.best_tri ||
                                              (tid == s.best_tri && (unsigned)s.inst_id < (unsigned)s.best_inst)));
}

// One triangle of the current leaf; returns true when it is the ray's new best hit.
template <bool ANY, bool MASKED, bool STATS>
__device__ __forceinline__ bool tri_step(const TraceArgs& a, TraceState& s, const uint4& r0, const uint4& r1,
                                         const uint4& r2) {
    const float4 v0 = as_float4(r0), v1 = as_float4(r1), v2 = as_float4(r2);
    if (STATS) s.ct++;
    float th = 0.0f, uh = 0.0f, vh = 0.0f;
    const int tid = (int)r1.w;
    bool better = tri_hit(s.cs, v0, v1, v2, th, uh, vh) && th >= s.tmin;
    better = better && is_better<ANY>(s, th, tid);
    if (MASKED && better) {
        const int op = texel_opaque(a, tid, uh, vh);
        if (op & 2) s.bad = 1;
        better = op & 1;
    }
    s.best_t = better ? th : s.best_t;
    s.best_u = better ? uh : s.best_u;
    s.best_tri = better ? tid : s.best_tri;
    s.best_inst = better ? s.inst_id : s.best_inst;
    return better;
}

// A ray whose subtree is done: the next instance of its leaf, or (back in world space if that
// was the last one) the top of the stack.  Returns false when the ray is finished.
template <typename POP>
__device__ __forceinline__ bool resume(TraceState& s, int sp, POP pop) {
    const bool exhausted = sp == s.inst_sp;
    const bool leave = exhausted && s.inst_next < 0;
    if (leave) {
        to_world(s);
        s.inst_sp = -1;
    }
    const bool again = exhausted && !leave;
    int link = ~s.inst_next;
    if (!again) {
        if (sp == 0) return false;
        link = pop();
    }
    s.kind = link >= 0 ? kNode : (again || s.inst_sp < 0) ? kInst : kTri;
    s.item = link >= 0 ? link : ~link;
    return true;
}

// The instance s.item: its record is fetched and the ray goes to its object space and root node.
template <bool STATS>
__device__ __forceinline__ void inst_step(const TraceArgs& a, TraceState& s, int sp) {
    const uint32_t i = (uint32_t)s.item;
    if (i < (uint32_t)a.n_inst) {
        const auto* p = gview(reinterpret_cast<const uint4*>(a.inst)) + 4u * (size_t)i;
        const uint4 r0 = p[0], r1 = p[1], r2 = p[2], r3 = p[3];
        s.item = enter_instance<STATS>(s, r0, r1, r2, r3, sp);
    } else {
        s.item = -1;  // fails the node's bounds check
        s.inst_next = -1;
    }
    s.kind = kNode;
}

// Where a node's link leads: an inner node, the first instance of a top-level leaf or the first
// triangle of a mesh leaf.
__device__ __forceinline__ void follow(TraceState& s, int link) {
    s.kind = link >= 0 ? kNode : link == kNoNode ? kNone : s.inst_sp < 0 ? kInst : kTri;
    s.item = link >= 0 ? link : ~link;
}

// Advances one ray by one step; returns true when the ray is finished.
//
// A step's time is its instructions, not its loads: with one wave per SIMD a step of the
// quantized tree took about 1,400 cycles of issue and 500 of load latency, and every kind of
// record that any lane of the wave is at costs the whole wave its code.  So each kind's code
// appears once per step, and a step takes a ray as far as one pass over that code can:
//   4-wide trees  one triangle, then (if that ended the leaf) the next thing off the stack, an
//                 instance entry and a node.  A ray's steps are its nodes plus the triangles after
//                 the first of a leaf.  Postponing triangles or instances until more lanes
//                 of the wave hold one made every workload slower (13-60%): a wave lasts as long
//                 as its longest ray.
//   BVH2          an instance entry, then one triangle or one node, whose records are loaded
//                 together.  Nodes are cheap here and twice as many, so a second load latency in
//                 the step costs more than the steps it saves (1M primary rays over 65K triangles:
//                 440 us against 553 us).
// MI355X, us per launch before (an instance entry and a pop in three places, one node or
// triangle per step) -> now: 1M primary rays, 65K triangles, quantized 551 -> 360, BVH2 590 ->
// 438; 300K diffuse rays, 250K triangles, quantized 537 -> 385; 200K rays over masked, rotated
// instances, quantized 1,216 -> 809; any hit, 1M shadow rays, BVH2 820 -> 653.
template <int BLOCK, int STACK_LDS, bool ANY, bool MASKED, bool STATS, int TREE>
__device__ __forceinline__ bool advance(const TraceArgs& a, TraceState& s, LaneStack<BLOCK, STACK_LDS>& st) {
    if constexpr (TREE != 0) {
        if (s.kind == kTri) {
            bool end = true;
            if (s.item < a.n_tris4 - 2) {
                const auto* p = gview(reinterpret_cast<const uint4*>(a.tris)) + (size_t)(uint32_t)s.item;
                const uint4 r0 = p[0], r1 = p[1], r2 = p[2];
                const bool better = tri_step<ANY, MASKED, STATS>(a, s, r0, r1, r2);
                if (ANY && better) return true;
                end = r2.w == kLeafEnd;
            } else {
                s.bad = 1;
            }
            s.item += 3;
            s.kind = end ? kNone : kTri;
        }
        if (s.kind == kNone && !resume(s, st.sp, [&] { return st.pop(); })) return true;
        if (s.kind == kInst) inst_step<STATS>(a, s, st.sp);
        if (s.kind == kNode) {
            int next = kNoNode;
            if ((uint32_t)s.item < (uint32_t)a.n_nodes) {
                const auto* p = gview(reinterpret_cast<const uint4*>(a.nodes)) +
                                (TREE == 1 ? 8u : 4u) * (size_t)(uint32_t)s.item;
                const uint4 r0 = p[0], r1 = p[1], r2 = p[2], r3 = p[3];
                if constexpr (TREE == 2) next = node_step4q<BLOCK, STACK_LDS, STATS>(s, st, r0, r1, r2, r3);
                else next = node_step4<BLOCK, STACK_LDS, STATS>(a, s, st, r0, r1, r2, r3);
            } else {
                s.bad = 1;
            }
            follow(s, next);
        }
        return false;
    } else {
        if (s.kind == kInst) inst_step<STATS>(a, s, st.sp);
        const int kind = s.kind;
        const char* base = (const char*)(kind == kNode ? a.nodes : a.tris);
        const uint32_t limit = (uint32_t)(kind == kNode ? a.n_nodes : max(a.n_tris4 - 2, 0));
        const int shift = kind == kTri ? 4 : 6;
        const bool ok = (uint32_t)s.item < limit;
        uint4 r0, r1, r2, r3;
        if (ok) {
            const auto* p = gview(reinterpret_cast<const uint4*>(base + ((uint64_t)(uint32_t)s.item << shift)));
            r0 = p[0]; r1 = p[1]; r2 = p[2];
            if (kind == kNode) r3 = p[3];
        }
        __builtin_amdgcn_sched_barrier(0);
        int next = kNoNode;  // link to go on with, or
        bool list = false;   // the next triangle of the leaf
        if (!ok) {
            s.bad = 1;
        } else if (kind == kTri) {
            const bool better = tri_step<ANY, MASKED, STATS>(a, s, r0, r1, r2);
            if (ANY && better) return true;
            list = r2.w != kLeafEnd;
        } else {
            next = node_step2<BLOCK, STACK_LDS, STATS>(s, st, r0, r1, r2, r3);
        }
        const int item = s.item + 3;
        follow(s, next);
        s.kind = list ? kTri : s.kind;
        s.item = list ? item : s.item;
        return s.kind == kNone && !resume(s, st.sp, [&] { return st.pop(); });
    }
}

template <int BLOCK, int STACK_LDS>
__device__ __forceinline__ void stack_init(LaneStack<BLOCK, STACK_LDS>& st, int* lds, const TraceArgs& a) {
    st.lds = lds;
    st.spill = a.spill;
    st.spill_depth = a.spill_depth;
    st.lane_slot = threadIdx.x;
    st.spill_slot = blockIdx.x * BLOCK + threadIdx.x;
    st.spill_stride = a.spill_stride;
    st.sp = 0;
}

// ---------------------------------------------------------------------------------------
// Four lanes per ray (quantized tree).  The lanes of a quad hold the same ray and go through the
// same steps; lane j tests child box j of a node and triangle j of a leaf, and the quad sorts with
// DPP exchanges.  A step is then about half the instructions of one with a lane per ray.
// Visiting order, and so every hit, is that of `advance`.
//
// Small queues start that way (quad_trace): a wave lasts as long as the longest of 16 rays
// instead of 64, and a queue that would leave SIMDs with one wave or none spreads over four times
// the waves.  The stack of such a quad has the LDS of its four lanes.
// MI355X, us per launch, one lane -> four lanes per ray, quantized tree, 65K triangles: 1,000
// diffuse rays 186 -> 111, 16,000: 209 -> 116, 65,000: 216 -> 153, 130,000: 203 -> 243; primary
// rays 16,000: 167 -> 95, 130,000: 162 -> 133; shadow rays 65,000: 156 -> 122, 130,000: 161 ->
// 187; 1M primary rays 360 -> 694 (the chip is full and four lanes do more work per ray).
//
// Waves of larger queues start with a lane per ray and go over to it (wave_trace): with 37% (1M
// primary rays) to 23% (diffuse rays) of the lanes busy on average without that, most steps of a wave
// serve few rays (with it 46% for the primary rays).  Moving the state costs about one step.  us per launch before -> now: 1M primary rays
// 361 -> 353, 1M shadow rays 534 -> 486, 300K diffuse rays over 250K triangles 397 -> 334, 200K rays
// over masked instances 790 -> 743, 48 queues in a batch 1,040 -> 917; path-traced frame 640x480
// 4,261 -> 4,002.

// Stack entries written before are read after by other lanes of the wave.  The hardware keeps a
// wave's accesses to one address in order, in LDS and in memory; this holds the compiler to it.
__device__ __forceinline__ void stack_shared() {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// Lane (4 q + k) receives the value of lane 4 q + {A, B, C, D}[k].
template <int A, int B, int C, int D>
__device__ __forceinline__ uint32_t quad_u(uint32_t v) {
    return (uint32_t)__builtin_amdgcn_update_dpp((int)v, (int)v, A | (B << 2) | (C << 4) | (D << 6), 0xF, 0xF, false);
}
template <int A, int B, int C, int D>
__device__ __forceinline__ float quad_f(float v) {
    return __uint_as_float(quad_u<A, B, C, D>(__float_as_uint(v)));
}

// Compare-exchange of (distance, link) between the lanes of a pair, as order2: the pair's low lane
// keeps the nearer, its own on a tie.
template <int A, int B, int C, int D>
__device__ __forceinline__ void quad_order(float& d, uint32_t& c, bool low) {
    const float od = quad_f<A, B, C, D>(d);
    const uint32_t oc = quad_u<A, B, C, D>(c);
    const bool take = low ? od < d : d < od;
    d = take ? od : d;
    c = take ? oc : c;
}

// A candidate hit of the lane against that of another lane of the quad: the smaller (t, triangle
// id), or for any hit the earlier one of the list (from = lane + 1, 0: no candidate).
struct Candidate {
    float t, u;
    uint32_t tri, from;
};
template <bool ANY, int A, int B, int C, int D>
__device__ __forceinline__ void quad_best(Candidate& c) {
    const float t = quad_f<A, B, C, D>(c.t), u = quad_f<A, B, C, D>(c.u);
    const uint32_t tri = quad_u<A, B, C, D>(c.tri), from = quad_u<A, B, C, D>(c.from);
    const bool nearer = ANY ? from < c.from : t < c.t || (t == c.t && (tri < c.tri || (tri == c.tri && from < c.from)));
    const bool take = from != 0 && (c.from == 0 || nearer);
    c.t = take ? t : c.t;
    c.u = take ? u : c.u;
    c.tri = take ? tri : c.tri;
    c.from = take ? from : c.from;
}

// One step of a quad's ray, as `advance` for the quantized tree; j is the lane's place in the quad.
template <bool ANY, bool MASKED, typename STACK>
__device__ __forceinline__ bool advance_quad(const TraceArgs& a, TraceState& s, STACK& st, int j) {
    if (s.kind == kTri) {
        const int t = s.item + 3 * j;
        const bool in = t < a.n_tris4 - 2;
        uint4 r0 = {}, r1 = {}, r2 = {};
        r2.w = kLeafEnd;
        if (in) {
            const auto* p = gview(reinterpret_cast<const uint4*>(a.tris)) + (size_t)(uint32_t)t;
            r0 = p[0]; r1 = p[1]; r2 = p[2];
        }
        // the triangles after the leaf's last one belong to another leaf
        const uint32_t e = r2.w == kLeafEnd ? 1u : 0u;
        const uint32_t e0 = quad_u<0, 0, 0, 0>(e), e1 = quad_u<1, 1, 1, 1>(e), e2 = quad_u<2, 2, 2, 2>(e),
                       e3 = quad_u<3, 3, 3, 3>(e);
        const bool mine = !((j > 0 && e0) || (j > 1 && e1) || (j > 2 && e2));
        if (mine && !in) s.bad = 1;
        float th = 0.0f, uh = 0.0f, vh = 0.0f;
        const uint32_t tid = r1.w;
        bool better = mine && in && tri_hit(s.cs, as_float4(r0), as_float4(r1), as_float4(r2), th, uh, vh) &&
                      th >= s.tmin;
        better = better && is_better<ANY>(s, th, (int)tid);
        if (MASKED && better) {
            const int op = texel_opaque(a, (int)tid, uh, vh);
            if (op & 2) s.bad = 1;
            better = op & 1;
        }
        if (__ballot(better)) {
            Candidate c{th, uh, tid, better ? (uint32_t)j + 1u : 0u};
            quad_best<ANY, 1, 0, 3, 2>(c);
            quad_best<ANY, 2, 3, 0, 1>(c);
            const bool hit = c.from != 0;
            s.best_t = hit ? c.t : s.best_t;
            s.best_u = hit ? c.u : s.best_u;
            s.best_tri = hit ? (int)c.tri : s.best_tri;
            s.best_inst = hit ? s.inst_id : s.best_inst;
            if (ANY && hit) return true;
        }
        s.item += 12;
        s.kind = (e0 | e1 | e2 | e3) ? kNone : kTri;
    }
    if (s.kind == kNone && !resume(s, st.sp, [&] { return st.pop(); })) return true;
    if (s.kind == kInst) inst_step<false>(a, s, st.sp);
    if (s.kind == kNode) {
        int next = kNoNode;
        const uint32_t n = (uint32_t)s.item;
        if (n < (uint32_t)a.n_nodes) {
            const auto* p = gview(reinterpret_cast<const uint4*>(a.nodes)) + 4u * (size_t)n;
            const uint4 w0 = p[0], w2 = p[2];
            const uint2 w3 = gview(reinterpret_cast<const uint2*>(a.nodes))[8u * (size_t)n + 6];
            uint32_t c = gview(reinterpret_cast<const uint32_t*>(a.nodes))[16u * (size_t)n + 4 + j];
            // byte j of the low and of the high word of an axis, near one first (see node_step4q)
            const uint32_t lo_hi = (uint32_t)(j | (4 + j) << 8), hi_lo = (uint32_t)((4 + j) | j << 8);
            const uint32_t bx = __builtin_amdgcn_perm(w2.y, w2.x, s.cs.idx >= 0.0f ? lo_hi : hi_lo);
            const uint32_t by = __builtin_amdgcn_perm(w2.w, w2.z, s.cs.idy >= 0.0f ? lo_hi : hi_lo);
            const uint32_t bz = __builtin_amdgcn_perm(w3.y, w3.x, s.cs.idz >= 0.0f ? lo_hi : hi_lo);
            float d;
            const bool h = quant_box_hit(s, QuantFrame(w0), bx, 0, bx, 1, by, 0, by, 1, bz, 0, bz, 1, d) && c > n;
            d = h ? d : __int_as_float(0x7f800000);
            const uint32_t one = h ? 1u : 0u;
            uint32_t cnt = one + quad_u<1, 0, 3, 2>(one);
            cnt += quad_u<2, 3, 0, 1>(cnt);
            // the sorting network of descend4
            quad_order<1, 0, 3, 2>(d, c, !(j & 1));
            quad_order<2, 3, 0, 1>(d, c, j < 2);
            quad_order<0, 2, 1, 3>(d, c, j < 2);
            const int top = st.sp + max((int)cnt - 1, 0);
            if (st.holds(top)) {
                if (j > 0 && (uint32_t)j < cnt) st.put(top - j, (int)c);
                stack_shared();
                st.sp = top;
            } else {
                s.bad = 1;  // not for the trees the launch was checked for
            }
            next = cnt ? (int)quad_u<0, 0, 0, 0>(c) : kNoNode;
        } else {
            s.bad = 1;
        }
        follow(s, next);
    }
    return false;
}

template <bool STATS>
__device__ __forceinline__ void write_result(const TraceArgs& a, const TraceState& s, int id) {
    gview_w(a.hits)[id] = make_int4(s.best_tri, s.best_inst, __float_as_int(s.best_t), __float_as_int(s.best_u));
    if (STATS && a.counts) {
        a.counts[3 * (size_t)id + 0] = s.cn;
        a.counts[3 * (size_t)id + 1] = s.ct;
        a.counts[3 * (size_t)id + 2] = s.ci;
    }
    if (STATS && a.depth_hist) atomicAdd(&a.depth_hist[min(s.cd, 63u)], 1u);
    if (s.bad) atomicAdd(a.err, 1);
}

// Writes the result of a quad's ray.
__device__ __forceinline__ void write_quad(const TraceArgs& a, TraceState& s, int id, int j) {
    s.bad |= (int)quad_u<1, 0, 3, 2>((uint32_t)s.bad);
    s.bad |= (int)quad_u<2, 3, 0, 1>((uint32_t)s.bad);
    if (j == 0) write_result<false>(a, s, id);
}

// Traces ray `id` with this thread's quad.
template <int BLOCK, int STACK_LDS, bool ANY, bool MASKED>
__device__ __forceinline__ void quad_trace(const TraceArgs& a, int* lds_stack, int id) {
    const int j = threadIdx.x & 3;
    TraceState s;
    state_init(s, gview(a.rays)[2 * (size_t)id], gview(a.rays)[2 * (size_t)id + 1], a.root);
    QuadStack<BLOCK, STACK_LDS> st{lds_stack + (threadIdx.x >> 2), 0};
    while (!advance_quad<ANY, MASKED>(a, s, st, j)) {
    }
    write_quad(a, s, id, j);
}

__device__ __forceinline__ void from_lane(int& v, int lane) { v = __builtin_amdgcn_ds_bpermute(4 * lane, v); }
__device__ __forceinline__ void from_lane(float& v, int lane) {
    v = __int_as_float(__builtin_amdgcn_ds_bpermute(4 * lane, __float_as_int(v)));
}

// Traces the wave's rays (ray `id` of every lane with `valid`; whole waves call it), one per lane
// until at most 16 are left, those with a quad of lanes each.
template <int BLOCK, int STACK_LDS, bool ANY, bool MASKED>
__device__ __forceinline__ void wave_trace(const TraceArgs& a, LaneStack<BLOCK, STACK_LDS>& st, int id, bool valid) {
    const int lane = threadIdx.x & 63;
    TraceState s;
    const int at = valid ? id : 0;
    state_init(s, gview(a.rays)[2 * (size_t)at], gview(a.rays)[2 * (size_t)at + 1], a.root);
    st.sp = 0;
    bool live = valid;
    unsigned long long left = __ballot(live);
    while (__popcll(left) > 16) {
        if (live && advance<BLOCK, STACK_LDS, ANY, MASKED, false, 2>(a, s, st)) {
            write_result<false>(a, s, id);
            live = false;
        }
        left = __ballot(live);
    }
    if (!left) return;
    // the r-th ray left goes to quad r: its lane's number to lane 4 r (the other lanes' to a lane
    // that no one asks), then to the quad, which takes over its state and its stack
    const int rank = __builtin_amdgcn_mbcnt_hi((unsigned)(left >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)left, 0u));
    const int from = (int)quad_u<0, 0, 0, 0>((uint32_t)__builtin_amdgcn_ds_permute(4 * (live ? 4 * rank : 1), lane));
    const int j = lane & 3;
    live = (lane >> 2) < __popcll(left);
    from_lane(s.world.ox, from); from_lane(s.world.oy, from); from_lane(s.world.oz, from);
    from_lane(s.world.dx, from); from_lane(s.world.dy, from); from_lane(s.world.dz, from);
    from_lane(s.world.idx, from); from_lane(s.world.idy, from); from_lane(s.world.idz, from);
    from_lane(s.cs.ox, from); from_lane(s.cs.oy, from); from_lane(s.cs.oz, from);
    from_lane(s.cs.dx, from); from_lane(s.cs.dy, from); from_lane(s.cs.dz, from);
    from_lane(s.cs.idx, from); from_lane(s.cs.idy, from); from_lane(s.cs.idz, from);
    s.cs.oidx = s.cs.ox * s.cs.idx; s.cs.oidy = s.cs.oy * s.cs.idy; s.cs.oidz = s.cs.oz * s.cs.idz;
    from_lane(s.tmin, from); from_lane(s.best_t, from); from_lane(s.best_u, from);
    from_lane(s.best_tri, from); from_lane(s.best_inst, from);
    from_lane(s.kind, from); from_lane(s.item, from);
    from_lane(s.inst_id, from); from_lane(s.inst_next, from); from_lane(s.inst_sp, from);
    from_lane(s.bad, from); from_lane(st.sp, from); from_lane(id, from);
    LaneStack<BLOCK, STACK_LDS> theirs = st;
    theirs.lane_slot += from - lane;
    theirs.spill_slot += from - lane;
    stack_shared();
    while (__ballot(live)) {
        if (live && advance_quad<ANY, MASKED>(a, s, theirs, j)) {
            write_quad(a, s, id, j);
            live = false;
        }
    }
}

// Waves per SIMD a traversal kernel is held to: 8 over the BVH2 (64 VGPRs), 7 over the 4-wide tree
// (72), 6 over the quantized one (80: both mappings of rays to lanes without scratch; held to 7 its
// 24 bytes of scratch per lane cost batches 5% and frames 1.5%).
constexpr int min_waves(int tree) { return tree == 0 ? 8 : tree == 1 ? 7 : 6; }

// One ray per thread (rays strided over the grid when it is smaller than the ray count), or four
// lanes per ray when the launch holds at most a.quad rays (the host then sizes the grid for four
// threads per ray and has checked the stack).
template <int BLOCK, int STACK_LDS, bool ANY, bool MASKED, bool STATS, int TREE>
__global__ __launch_bounds__(BLOCK, STATS ? 1 : min_waves(TREE)) void k_trace(TraceArgs a) {
    __shared__ int lds_stack[STACK_LDS * BLOCK];
    const int count = launch_count(a);
    if constexpr (TREE == 2 && !STATS) {
        if (count <= a.quad) {
            const int id = (int)(blockIdx.x * BLOCK + threadIdx.x) >> 2;
            if (id < count) quad_trace<BLOCK, STACK_LDS, ANY, MASKED>(a, lds_stack, id);
            return;
        }
    }
    if ((int)(blockIdx.x * BLOCK) >= count) return;  // sized for the capacity of a device-side count
    LaneStack<BLOCK, STACK_LDS> st;
    stack_init(st, lds_stack, a);
    const int stride = gridDim.x * BLOCK;
    if constexpr (TREE == 2 && !STATS) {
        for (int first = blockIdx.x * BLOCK + (threadIdx.x & ~63); first < count; first += stride) {
            const int id = first + (threadIdx.x & 63);
            wave_trace<BLOCK, STACK_LDS, ANY, MASKED>(a, st, id, id < count);
        }
        return;
    }
    for (int id = blockIdx.x * BLOCK + threadIdx.x; id < count; id += stride) {
        TraceState s;
        state_init(s, a.rays[2 * (size_t)id], a.rays[2 * (size_t)id + 1], a.root);
        st.sp = 0;
        while (!advance<BLOCK, STACK_LDS, ANY, MASKED, STATS, TREE>(a, s, st)) {
        }
        write_result<STATS>(a, s, id);
    }
}

// Persistent variant: every wave keeps 64 rays in flight and, whenever at least `refill` of its
// lanes have finished, takes the next consecutive block of ray ids for them with one atomic
// on a global counter (ballot + popcount + mbcnt).  Each iteration advances every active lane
// by one step of `advance`, so the per-ray results are those of k_trace.
// counter[0] = next ray, counter[1] = finished waves; the last wave to finish resets both.
template <int BLOCK, int STACK_LDS, bool ANY, bool MASKED, bool STATS, int TREE>
__global__ __launch_bounds__(BLOCK) void k_trace_dyn(TraceArgs a, int refill) {
    __shared__ int lds_stack[STACK_LDS * BLOCK];
    LaneStack<BLOCK, STACK_LDS> st;
    stack_init(st, lds_stack, a);
    const int lane = __lane_id();
    int* counter = a.work_counter;
    int id = -1;             // ray of this lane, -1 = none
    bool exhausted = false;  // wave-uniform: no rays left to fetch
    const int count = launch_count(a);
    TraceState s;
    for (;;) {
        const unsigned long long idle = __ballot(id < 0);
        if (!exhausted && __popcll(idle) >= refill) {
            const int n = __popcll(idle);
            const int leader = __ffsll((long long)idle) - 1;
            int base = 0;
            if (lane == leader) base = atomicAdd(&counter[0], n);
            base = __shfl(base, leader, 64);
            if (base + n >= count) exhausted = true;
            if (id < 0) {
                const int r = base + __builtin_amdgcn_mbcnt_hi((unsigned)(idle >> 32),
                                                               __builtin_amdgcn_mbcnt_lo((unsigned)idle, 0u));
                if (r < count) {
                    id = r;
                    state_init(s, a.rays[2 * (size_t)r], a.rays[2 * (size_t)r + 1], a.root);
                    st.sp = 0;
                }
            }
        }
        if (__ballot(id >= 0) == 0) {
            if (exhausted) break;
            continue;
        }
        if (id >= 0 && advance<BLOCK, STACK_LDS, ANY, MASKED, STATS, TREE>(a, s, st)) {
            write_result<STATS>(a, s, id);
            id = -1;
        }
    }
    // the last wave out resets the counters for the launch that reuses this slot
    if (lane == 0) {
        const int waves = gridDim.x * (BLOCK / 64);
        if (atomicAdd(&counter[1], 1) == waves - 1) {
            atomicExch(&counter[0], 0);
            atomicExch(&counter[1], 0);
        }
    }
}

// ---------------------------------------------------------------------------------------
// Batched traversal: many ray queues, each with its own scene, in one launch per kernel
// variant.  The queues of a launch are cut into chunks of 64 consecutive rays; every wave
// takes the next chunk from a global counter, finds its queue by binary search over the
// queues' first chunks (wave-uniform, so the queue's arguments sit in scalar registers) and
// traces one ray per lane with the same per-ray steps as k_trace, so every queue's hits are
// those of a launch of its own.
struct BatchItem {
    TraceArgs a;           // a.count: rays of this launch (set by k_batch_prefix)
    const int* count_dev;  // device ray count read when the launch runs, or null
    int capacity;          // rays (count_dev null) or the upper bound of *count_dev
    int chunk_begin;       // first chunk of this queue within its launch group
    int group;             // launch group: 2 * any_hit + masked
};

struct BatchGroups {
    int first[5];  // items of group g: [first[g], first[g + 1])
};

// One block of 1024 threads: ray counts of this launch, each queue's first chunk, chunks per group.
__global__ __launch_bounds__(1024) void k_batch_prefix(BatchItem* items, BatchGroups groups, int* group_chunks) {
    // thread t owns the queues [b0, b1); items are ordered by group, so a queue's chunk_begin is
    // its exclusive chunk prefix over all queues minus that of its group's first queue
    __shared__ int part[1024];
    __shared__ int base[5];
    const int n_items = groups.first[4];
    const int t = threadIdx.x;
    const int per = (n_items + 1023) / 1024;
    const int b0 = min(n_items, t * per), b1 = min(n_items, b0 + per);
    int sum = 0;
    for (int i = b0; i < b1; i++) {
        int n = items[i].capacity;
        if (items[i].count_dev) n = min(max(*items[i].count_dev, 0), n);
        items[i].a.count = n;
        sum += (n + 63) >> 6;
    }
    part[t] = sum;
    __syncthreads();
    for (int d = 1; d < 1024; d <<= 1) {  // inclusive scan of the per-thread sums
        const int v = t >= d ? part[t - d] : 0;
        __syncthreads();
        part[t] += v;
        __syncthreads();
    }
    const int total = part[1023];
    int run = part[t] - sum;  // exclusive prefix at b0
    for (int i = b0; i < b1; i++) {
        for (int g = 0; g < 5; g++)
            if (groups.first[g] == i) base[g] = run;
        run += (items[i].a.count + 63) >> 6;
    }
    __syncthreads();
    run = part[t] - sum;
    int g = 0;
    for (int i = b0; i < b1; i++) {
        while (g < 3 && groups.first[g + 1] <= i) g++;
        items[i].chunk_begin = run - base[g];
        run += (items[i].a.count + 63) >> 6;
    }
    if (t < 4) {
        const int f0 = groups.first[t], f1 = groups.first[t + 1];
        group_chunks[t] = f0 == f1 ? 0 : (f1 < n_items ? base[t + 1] : total) - base[t];
    }
}

// QUADS (quantized tree): four lanes per ray, a wave taking a quarter of a chunk at a time.  A
// kernel of its own: both mappings in one kernel cost the one-lane mapping 7% (48 queues, 1.3M
// rays: 1,157 us against 1,082).  Where the queue sizes are only known on the device both kernels
// are launched and `limit` chunks decide which of them works: the one-lane kernel above it, the
// other up to it (limit < 0: the one-lane kernel always).
template <int BLOCK, int STACK_LDS, bool ANY, bool MASKED, int TREE, bool QUADS>
__global__ __launch_bounds__(BLOCK, min_waves(TREE)) void k_trace_batch(
    const BatchItem* __restrict__ items, int first, int n_items, const int* __restrict__ total_chunks, int* counter,
    int* spill, int spill_depth, int limit) {
    __shared__ int lds_stack[STACK_LDS * BLOCK];
    LaneStack<BLOCK, STACK_LDS> st;
    st.lds = lds_stack;
    st.spill = spill;
    st.spill_depth = spill_depth;
    st.lane_slot = threadIdx.x;
    st.spill_slot = blockIdx.x * BLOCK + threadIdx.x;
    st.spill_stride = gridDim.x * BLOCK;
    st.sp = 0;
    const int lane = __lane_id();
    const int chunks = __builtin_amdgcn_readfirstlane(*total_chunks);
    if (QUADS ? chunks > limit : chunks <= limit) return;  // the same for the whole grid: counters untouched
    const int total = QUADS ? 4 * chunks : chunks;  // pieces of 16 or 64 rays
    for (;;) {
        int piece = 0;
        if (lane == 0) piece = atomicAdd(&counter[0], 1);
        piece = __builtin_amdgcn_readfirstlane(__shfl(piece, 0, 64));
        if (piece >= total) break;
        const int c = QUADS ? piece >> 2 : piece;
        // the queue owning chunk c: the last one whose first chunk is <= c (queues without
        // rays share their first chunk with the next queue and are skipped)
        int lo = first, hi = first + n_items - 1;
        while (lo < hi) {
            const int mid = (lo + hi + 1) >> 1;
            if (__builtin_amdgcn_readfirstlane(items[mid].chunk_begin) <= c) lo = mid;
            else hi = mid - 1;
        }
        lo = __builtin_amdgcn_readfirstlane(lo);
        const TraceArgs a = items[lo].a;
        const int begin = (c - items[lo].chunk_begin) * 64;
        if constexpr (QUADS) {
            const int id = begin + (piece & 3) * 16 + (lane >> 2);
            if (id < a.count) quad_trace<BLOCK, STACK_LDS, ANY, MASKED>(a, lds_stack, id);
        } else {
            const int id = begin + lane;
            if constexpr (TREE == 2) {
                wave_trace<BLOCK, STACK_LDS, ANY, MASKED>(a, st, id, id < a.count);
            } else if (id < a.count) {
                TraceState s;
                state_init(s, gview(a.rays)[2 * (size_t)id], gview(a.rays)[2 * (size_t)id + 1], a.root);
                st.sp = 0;
                while (!advance<BLOCK, STACK_LDS, ANY, MASKED, false, TREE>(a, s, st)) {
                }
                write_result<false>(a, s, id);
            }
        }
    }
    if (lane == 0) {
        const int waves = gridDim.x * (BLOCK / 64);
        if (atomicAdd(&counter[1], 1) == waves - 1) {
            atomicExch(&counter[0], 0);
            atomicExch(&counter[1], 0);
        }
    }
}

}  // namespace imba
