// trace.hip — ray traversal and shading, replacing optixLaunch of raygen_program
// (plugins/optix_hpg/src/optix/AbstractRenderer.cpp:106, cuda_resources/raygen.cu:79-278) and the
// intersection / closest-hit programs (cuda_resources/sphere.cuh:43-57, 94-131).
//
// Launch shape: a persistent grid (at most blocks_per_cu x CUs blocks of 256 threads). Each wavefront
// takes 8x8-pixel tiles from work queues until none are left; a lane owns one pixel and loops over
// its samples in order, so the per-pixel random stream is the reference's one (TEA seed, two LCG
// draws per sample for the jitter).
//
// Traversal: BVH2 with both child boxes in the 64-byte node (four 16-byte loads per visit),
// ordered front-to-back, the spheres of a leaf reference tested apart from the node visits, two at
// a time (leaf pairs); the samples of one pixel walk the tree together with scalar loads. The
// traversal stack keeps its lowest S entries in LDS (lane-strided, conflict free) and spills deeper
// ones to a per-lane global region. Closest hit keeps the lowest particle ID among equal t; boxes
// whose entry distance equals the current best are still visited so that ties resolve the same way
// whatever the visiting order. AO rays stop at the first occluder (any hit).
#include <float.h>

#include <algorithm>
#include <cstring>

#include "ctx.hpp"

namespace mmhrt {
namespace {

constexpr int TB = 256;                  // threads per block

struct TraceArgs {
    const Node* nodes;
    const float4* leaf_sph;
    const uint32_t* leaf_id;
    const float4* col;
    const SceneInfo* info;
    int32_t* spill;
    uint32_t spill_stride;  // lanes in the grid
    uint32_t* ctr;          // [1] overflow flag, [2..9] u64 counters, from TRACE_QUEUE on the work queues
    uint32_t n_tiles, tiles_x;
    uint32_t sub_log2;      // k_trace_sl: a unit of work is 1 / (1 << sub_log2) of a tile's passes
    uint32_t tw_log2;  // pixel tile = (1 << tw_log2) x (64 >> tw_log2), one wavefront
    float4* out_col;
    float* out_depth;
    float* out_t;
    int32_t* out_id;
    uint32_t* out_rgba8;
    __half* out_aux;
    FrameConsts fc;
    // treelet P-k-d trees (nodes then hold the top tree over the treelets)
    const uint8_t* pkd_dim;  // split axis of the node at each position
    const float* tl_rmax;    // largest radius of each treelet
    uint32_t n_sph;          // spheres
    uint32_t tl_log2;        // log2 of the treelet size
    const uint32_t* order;   // k_trace over treelets: the tiles, the dearest first (null: as they lie)
};

// The units of work of a launch (tiles, or parts of them), dealt in 8 contiguous bands, one queue
// per band. A wavefront's first unit is fixed by its number, later ones come from the counter of its
// own band's queue (workgroups go to the 8 XCDs in turn, so a band stays with one XCD's L2), and when
// that is used up from the other bands. Every taken unit used to be one atomic on one counter, and
// those run one after the other, about 10 ns each: 8192 wavefronts that each find out that nothing is
// left took 90 us by themselves (a 320x240 frame traced in 188 us, in 99 us with fixed tiles), and the
// refills of a 1080p frame 0.5 ms. All lanes of the wavefront call grab() together.
struct WorkQueue {
    uint32_t* q;      // counter of queue k at q[k * TRACE_QUEUE_STRIDE]: units taken beyond the fixed first ones
    uint32_t total;   // units
    uint32_t per;     // units per band
    uint32_t k;       // the queue this wavefront takes from
    bool first;
    __device__ __forceinline__ WorkQueue(uint32_t* ctr, uint32_t units)
        : q(ctr + TRACE_QUEUE), total(units), per((units + 7u) / 8u), k(blockIdx.x & 7u), first(true) {}
    __device__ __forceinline__ uint32_t size(uint32_t b) const {
        const uint32_t lo = b * per;
        return lo >= total ? 0u : (total - lo < per ? total - lo : per);
    }
    // wavefronts whose own queue is b: those of the workgroups b, b + 8, ...
    __device__ __forceinline__ uint32_t owners(uint32_t b) const {
        return (gridDim.x + 7u - b) / 8u * (TB / 64);
    }
    // a unit's place when the bands' first units come first, then their second ones, ...
    __device__ __forceinline__ uint32_t rank(uint32_t u) const {
        const uint32_t b = u / per, i = u - b * per, full = total / per, part = total - full * per;
        return i * full + (part < i ? part : i) + (b < full ? b : full);
    }
    // the next unit, or 0xffffffff when all are taken
    __device__ __forceinline__ uint32_t grab() {
        if (first) {
            first = false;
            const uint32_t w = (blockIdx.x >> 3) * (TB / 64) + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
            if (w < size(k)) return k * per + w;
        } else {
            const uint32_t u = take(k);
            if (u != 0xffffffffu) return u;
        }
        for (;;) {  // another queue that has units left, the nearest one on; reads first, they do not queue up
            const uint32_t lane = __lane_id();
            const uint32_t b = (k + lane) & 7u;
            bool left = false;
            if (lane < 8u)
                left = owners(b) + __hip_atomic_load(q + b * TRACE_QUEUE_STRIDE, __ATOMIC_RELAXED,
                                                     __HIP_MEMORY_SCOPE_AGENT) < size(b);
            const uint64_t m = __ballot(left);
            if (!m) return 0xffffffffu;
            k = (k + (uint32_t)__ffsll((unsigned long long)m) - 1u) & 7u;
            const uint32_t u = take(k);
            if (u != 0xffffffffu) return u;
        }
    }
    __device__ __forceinline__ uint32_t take(uint32_t b) {
        uint32_t u = 0;
        if (__lane_id() == 0) u = atomicAdd(q + b * TRACE_QUEUE_STRIDE, 1u);
        u = __builtin_amdgcn_readfirstlane(u) + owners(b);
        return u < size(b) ? b * per + u : 0xffffffffu;
    }
};

// Reference of no node: the bottom of a stack. Not a leaf reference, whose k is below 2^31 - 1.
constexpr int32_t REF_NONE = INT32_MIN;

// Traversal stack of one lane: (reference, entry distance of its box), the lowest N entries in
// LDS, lane-interleaved. Deeper entries spill their reference alone to the lane's global words
// and come back with an entry distance below every ray's (they are visited without the test).
// With SPILL_DIST in S they spill both words: the treelets' shallow trees (at most 22 top levels
// and 10 inside a treelet) fit the lane's words that way.
// Entry 0 is a sentinel (REF_NONE, nearer than everything), so a pop needs no test for an empty stack,
// and the LDS accesses are 8 bytes through the LDS address space: with a pointer that could be to either
// memory the compiler merged the LDS read with that of a spilled entry into a flat load after an address
// select, on each pop's chain. The wavefront pops at one place per visit (a leaf put aside and a visit
// without a hit are the same loop). Trace kernel: 60M clustered spheres at 4K 5.75 ms, then 5.49; 50M
// FCC spheres at 1080p with AO, 1 sample 0.72, then 0.66, 64 samples 13.7, then 13.5; 8M treelets 6.9,
// then 6.1. N = 10 is the most that leaves room for eight workgroups per CU (20 KB each); with 9, 8
// (and the sentinel) the clusters take 5.58 and 5.51, the FCC spheres 13.8 and 13.9.
constexpr int SPILL_DIST = 256;
typedef int i32x2 __attribute__((ext_vector_type(2)));
typedef __attribute__((address_space(3))) i32x2* lds_i32x2;
template <int S>
struct LaneStack {
    static constexpr int N = S & (SPILL_DIST - 1);
    static constexpr int W = S & SPILL_DIST ? 2 : 1;  // words per spilled entry
    static constexpr int CAP = N + TRACE_SPILL_PER_LANE / W;
    lds_i32x2 lds;  // element k at lds[k * TB]
    int32_t* spill;
    uint32_t stride;
    int sp;
    uint32_t* overflow;
    __device__ __forceinline__ LaneStack(int2* shared, int32_t* sl, uint32_t st, uint32_t* ov)
        : lds((lds_i32x2)shared), spill(sl), stride(st), sp(1), overflow(ov) {}
    __device__ __forceinline__ void reset() {
        lds[0] = (i32x2){REF_NONE, (int)0xff800000u};
        sp = 1;
    }
    // on: this lane pushes
    __device__ __forceinline__ void push(bool on, int32_t ref, float tn) {
        if (__builtin_expect(on && sp >= N, 0)) {
            if (sp < CAP) {
                spill[(size_t)(W * (sp - N)) * stride] = ref;
                if (W == 2) spill[(size_t)(W * (sp - N) + 1) * stride] = __float_as_int(tn);
                ++sp;
            } else {
                *overflow = 1u;  // cannot happen for a valid tree; recorded, entry dropped
            }
            on = false;
        }
        if (on) {
            lds[sp * TB] = (i32x2){ref, __float_as_int(tn)};
            ++sp;
        }
    }
    // the top entry (the stack holds at least the sentinel)
    __device__ __forceinline__ i32x2 take() {
        --sp;
        i32x2 e = lds[(sp < N ? sp : N - 1) * TB];
        if (__builtin_expect(sp >= N, 0)) {
            e.x = spill[(size_t)(W * (sp - N)) * stride];
            e.y = W == 2 ? spill[(size_t)(W * (sp - N) + 1) * stride] : (int)0xff800000u;
        }
        return e;
    }
    // for the lanes with `on`: the topmost reference whose box starts no farther than t_best becomes the
    // node (REF_NONE when there is none), or, if it is a leaf and none is aside, the one aside, and the
    // next one the node
    __device__ __forceinline__ void pop(bool on, float t_best, int32_t& node, int32_t& leaf) {
        if (on) {
            for (;;) {
                i32x2 e;
                do {
                    e = take();
                } while (__int_as_float(e.y) > t_best);
                if (e.x >= 0 || e.x == REF_NONE || leaf != REF_NONE) {
                    node = e.x;
                    break;
                }
                leaf = e.x;
            }
        }
    }
};

struct RayPre {
    V3 o, d, inv, oil, oih;
};

__device__ __forceinline__ RayPre prep(V3 o, V3 d, float pad) {
    RayPre r;
    r.o = o;
    r.d = d;
    float dx = fabsf(d.x) < 1e-30f ? __builtin_copysignf(1e-30f, d.x) : d.x;
    float dy = fabsf(d.y) < 1e-30f ? __builtin_copysignf(1e-30f, d.y) : d.y;
    float dz = fabsf(d.z) < 1e-30f ? __builtin_copysignf(1e-30f, d.z) : d.z;
    r.inv = V3{1.0f / dx, 1.0f / dy, 1.0f / dz};
    // box widened by pad: (lo - pad - o) * inv = lo * inv - (o + pad) * inv
    r.oil = V3{(o.x + pad) * r.inv.x, (o.y + pad) * r.inv.y, (o.z + pad) * r.inv.z};
    r.oih = V3{(o.x - pad) * r.inv.x, (o.y - pad) * r.inv.y, (o.z - pad) * r.inv.z};
    return r;
}

// Slab test of one child box (lo, hi); returns the entry distance, or +inf when missed. Minima and maxima
// issue at half the rate of multiply-adds (0.57e12 against 1.05e12 wavefront instructions/s over the device)
// and take two thirds of it, but selects do too: the planes picked by the signs of the direction, lane by
// lane, made 64 samples with AO over 50M spheres 2.5 % slower.
__device__ __forceinline__ float slab(const RayPre& r, float lx, float ly, float lz, float hx, float hy, float hz,
                                      float tmin, float tmax) {
    float x0 = __builtin_fmaf(lx, r.inv.x, -r.oil.x), x1 = __builtin_fmaf(hx, r.inv.x, -r.oih.x);
    float y0 = __builtin_fmaf(ly, r.inv.y, -r.oil.y), y1 = __builtin_fmaf(hy, r.inv.y, -r.oih.y);
    float z0 = __builtin_fmaf(lz, r.inv.z, -r.oil.z), z1 = __builtin_fmaf(hz, r.inv.z, -r.oih.z);
    float tn = fmaxf(fmaxf(fminf(x0, x1), fminf(y0, y1)), fmaxf(fminf(z0, z1), tmin));
    float tf = fminf(fminf(fmaxf(x0, x1), fmaxf(y0, y1)), fminf(fmaxf(z0, z1), tmax));
    return tn <= tf ? tn : INFINITY;
}

struct Count {
    uint64_t visits = 0, tests = 0, rays = 0, pair_visits = 0;
};

// Traversal of the LBVH by one lane, in two alternating phases. The inner phase visits stored
// nodes (64 bytes, both child boxes); a lane that reaches a leaf reference puts it aside and goes
// on with the next node from its stack, and the phase ends when every lane has one aside or is
// out of nodes. The leaf phase then tests the spheres put aside. Testing the spheres inside the
// visits instead made nearly every visit of a wavefront run the whole sphere test (two square
// roots and divisions) for the few lanes that had reached a leaf.
// Every leaf reference ~k stands for the two spheres k and k + 1, one 32-byte read, whether the
// node over them was left out of the tree (a leaf pair) or ~k is a single leaf: one more sphere
// tested changes no result, since the result is that over all spheres, whatever was visited (the
// least t, ties to the lowest particle id; for an any-hit ray whether there is a hit at all).
// A stack entry keeps its box's entry distance, and one that lies beyond the best hit when its
// turn comes is dropped without a fetch.

// One visit: both child boxes against the ray. The near child becomes the node, a far one that is hit
// too goes to the stack. A leaf reference is put aside if the lane has none aside yet; then, and with
// no child hit, the node is the next one from the stack.
template <int S, bool COUNT>
__device__ __forceinline__ void visit(const TraceArgs& A, const RayPre& r, float tmin, float t_best, int32_t& node,
                                      int32_t& leaf, LaneStack<S>& st, Count& cnt) {
    const float4* q = reinterpret_cast<const float4*>(A.nodes + node);
    const float4 a = q[0], b = q[1], c = q[2];
    const int2 d = *reinterpret_cast<const int2*>(q + 3);
    if (COUNT) cnt.visits++;
    const float tn0 = slab(r, a.x, a.y, a.z, a.w, b.x, b.y, tmin, t_best);
    const float tn1 = slab(r, b.z, b.w, c.x, c.y, c.z, c.w, tmin, t_best);
    const bool first0 = tn0 <= tn1;
    const float tnear = first0 ? tn0 : tn1, tfar = first0 ? tn1 : tn0;
    node = first0 ? d.x : d.y;
    st.push(tfar != INFINITY, first0 ? d.y : d.x, tfar);
    const bool none = tnear == INFINITY;
    const bool put = !none && node < 0 && leaf == REF_NONE;
    if (put) leaf = node;
    st.pop(none || put, t_best, node, leaf);
}

// The part of sphere_t before its square root: false when that sphere reports no hit. (With b < 0
// q = b -+ sqrt(delta) is negative and min(c / q, q) too, whatever c is: no report.)
__device__ __forceinline__ bool sphere_near(const RayPre& r, float4 s, V3& oc, float& b, float& delta) {
    oc = V3{r.o.x - s.x, r.o.y - s.y, r.o.z - s.z};
    b = dot(neg(oc), r.d);
    const V3 tmp = V3{oc.x + b * r.d.x, oc.y + b * r.d.y, oc.z + b * r.d.z};
    delta = s.w * s.w - dot(tmp, tmp);
    return !(delta < 0.0f) && !(b < 0.0f);
}
// The rest of it.
__device__ __forceinline__ float sphere_far(V3 oc, float rr, float b, float delta, float tmin, float tmax) {
    const float c = dot(oc, oc) - rr;
    const float q = b + __builtin_copysignf(__builtin_sqrtf(delta), b);
    const float t = fminf(c / q, q);
    if (t < 0.0f) return -1.0f;
    return (t > tmin && t < tmax) ? t : -1.0f;
}

// The spheres k and k + 1 of leaf reference ~k. Most spheres fail the first part of the test, so
// the second part runs once for whichever sphere passes, and again only for a lane where both do.
// Closest hit (any false): t_best and best are updated. any: returns true at a hit of a sphere
// other than leaf `skip` (best and t_best stay).
template <bool COUNT>
__device__ __forceinline__ bool test_leaf(const TraceArgs& A, const RayPre& r, float tmin, float tmax, int32_t ref,
                                          int skip, bool any, float& t_best, int& best, Count& cnt) {
    const int k0 = ~ref;
    const int k1 = (uint32_t)k0 + 1u < A.n_sph ? k0 + 1 : k0;
    const float4 s0 = A.leaf_sph[k0], s1 = A.leaf_sph[k1];
    if (COUNT) {
        cnt.visits++;
        cnt.pair_visits++;
        cnt.tests += 2;
    }
    V3 oc0, oc1;
    float b0, b1, e0, e1;
    bool p0 = sphere_near(r, s0, oc0, b0, e0);
    bool p1 = sphere_near(r, s1, oc1, b1, e1);
    p0 = p0 && k0 != skip;
    p1 = p1 && k1 != skip;
    while (p0 || p1) {
        const int leaf = p0 ? k0 : k1;
        const float w = p0 ? s0.w : s1.w;
        const float t = sphere_far(V3{p0 ? oc0.x : oc1.x, p0 ? oc0.y : oc1.y, p0 ? oc0.z : oc1.z}, w * w, p0 ? b0 : b1,
                                   p0 ? e0 : e1, tmin, tmax);
        if (p0)
            p0 = false;
        else
            p1 = false;
        if (t >= 0.0f) {
            if (any) return true;
            if (t < t_best) {
                t_best = t;
                best = leaf;
            } else if (t == t_best && best >= 0 && A.leaf_id[leaf] < A.leaf_id[best]) {
                best = leaf;
            }
        }
    }
    return false;
}

// The inner phase: visits until at most 3/8 of the lanes that began it still look for a leaf to put
// aside. A lane with a second leaf waits, and where leaves are rare (clusters of sub-pixel spheres)
// the wait for the last lanes is long: 60M clustered spheres at 4K, 1 sample, 6.82 ms when the phase
// ran until no lane looked for one, 5.83, 5.71, 5.81 and 6.09 ms at 1/4, 1/2, 3/4 and 15/16 of the
// lanes (1M uniform spheres: 0.50 ms, then 0.46, 0.45, 0.47, 0.53).
template <int S, bool COUNT>
__device__ __forceinline__ void inner_phase(const TraceArgs& A, const RayPre& r, float tmin, float t_best,
                                            int32_t& node, int32_t& leaf, LaneStack<S>& st, Count& cnt) {
    const int few = (int)__popcll(__ballot(node >= 0)) * 3 / 8;
    while (node >= 0) {
        visit<S, COUNT>(A, r, tmin, t_best, node, leaf, st, cnt);
        if ((int)__popcll(__ballot(leaf == REF_NONE)) <= few) break;
    }
}

// Node and sphere words read at a wavefront-uniform address: through the constant address space, so
// that they arrive in scalar registers (the structure is written by earlier kernels only).
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef int i32x4 __attribute__((ext_vector_type(4)));
typedef const __attribute__((address_space(4))) f32x4* const_f32x4;
typedef const __attribute__((address_space(4))) i32x4* const_i32x4;

// The start of a walk whose rays begin alike, as the primary rays of a tile and the AO rays of a pixel
// do: the wavefront goes down from the root together, by scalar loads, while at least 3/4 of its lanes
// meet the child that most of them meet first, and pushes the other child with each lane's own entry
// distance (infinite where the lane misses it). From the first node that is left with fewer lanes, that
// is over a leaf, or where the LDS part of the stack is nearly full, each lane goes on by itself. At 1
// sample 60M clustered spheres at 4K take 5.45 -> 5.25 ms, at 64 samples with AO 50M FCC spheres 12.8 ->
// 12.2 ms (all lanes, half or 3/4 of them: the same within 0.5 %). Not for a path's bounces, which
// part at once: 16 passes over 1M spheres took 10 % longer with it.
template <int S, bool COUNT>
__device__ __forceinline__ void descend_together(const TraceArgs& A, const RayPre& r, float tmin, float t_best,
                                                 int32_t& node, int32_t& leaf, LaneStack<S>& st, Count& cnt) {
    int32_t u = 0;
    const int keep = max(1, (int)__popcll(__ballot(true)) * 3 / 4);
    int sp = 1;
    for (;;) {
        const_f32x4 q = (const_f32x4)(uintptr_t)(A.nodes + u);
        const f32x4 a = q[0], b = q[1], c = q[2];
        const i32x4 d = *(const_i32x4)(q + 3);
        if (COUNT) cnt.visits++;
        const float tn0 = slab(r, a.x, a.y, a.z, a.w, b.x, b.y, tmin, t_best);
        const float tn1 = slab(r, b.z, b.w, c.x, c.y, c.z, c.w, tmin, t_best);
        const bool first0 = tn0 <= tn1;
        const uint64_t m0 = __ballot(tn0 != INFINITY), m1 = __ballot(tn1 != INFINITY);
        const bool pick0 = 2 * __popcll(__ballot(first0) & (m0 | m1)) >= __popcll(m0 | m1);
        const int32_t ch = pick0 ? d.x : d.y;
        if (ch < 0 || sp >= LaneStack<S>::N - 2 || (int)__popcll(pick0 ? m0 : m1) < keep) {
            const float tnear = first0 ? tn0 : tn1, tfar = first0 ? tn1 : tn0;
            node = first0 ? d.x : d.y;
            st.sp = sp;
            st.push(tfar != INFINITY, first0 ? d.y : d.x, tfar);
            const bool none = tnear == INFINITY;
            const bool put = !none && node < 0;
            if (put) leaf = node;
            st.pop(none || put, t_best, node, leaf);
            return;
        }
        if (pick0 ? m1 : m0) {
            st.lds[sp * TB] = (i32x2){pick0 ? d.y : d.x, __float_as_int(pick0 ? tn1 : tn0)};
            ++sp;
        }
        u = ch;
    }
}

// The walk of each lane by itself from its node, leaf aside and stack on: the closest hit of the rest.
template <int S, bool COUNT>
__device__ __forceinline__ void finish_closest(const TraceArgs& A, const RayPre& r, float tmin, float tmax, int32_t node,
                                               int32_t leaf, float& t_best, int& best, LaneStack<S>& st, Count& cnt) {
    while (node != REF_NONE || leaf != REF_NONE) {
        inner_phase<S, COUNT>(A, r, tmin, t_best, node, leaf, st, cnt);
        while (leaf != REF_NONE) {
            test_leaf<COUNT>(A, r, tmin, tmax, leaf, -1, false, t_best, best, cnt);
            const bool more = node < 0;  // (REF_NONE, too: nothing aside then)
            leaf = more ? node : REF_NONE;
            st.pop(more && node != REF_NONE, t_best, node, leaf);
        }
    }
}

// Closest hit: returns the leaf index of the nearest reported intersection (or -1) and its t.
template <int S, bool COUNT, bool TOG>
__device__ int trace_closest(const TraceArgs& A, const RayPre& r, float tmin, float tmax, float& t_best,
                             LaneStack<S>& st, Count& cnt) {
    int best = -1;
    t_best = tmax;
    int32_t node = 0, leaf = REF_NONE;
    st.reset();
    if (TOG) descend_together<S, COUNT>(A, r, tmin, t_best, node, leaf, st, cnt);
    finish_closest<S, COUNT>(A, r, tmin, tmax, node, leaf, t_best, best, st, cnt);
    return best;
}

// Any hit in (tmin, tmax) ignoring leaf `skip`.
template <int S, bool COUNT>
__device__ bool trace_any(const TraceArgs& A, const RayPre& r, float tmin, float tmax, int skip, LaneStack<S>& st,
                          Count& cnt) {
    int32_t node = 0, leaf = REF_NONE;
    st.reset();
    float tb = tmax;
    int best = -1;
    descend_together<S, COUNT>(A, r, tmin, tmax, node, leaf, st, cnt);
    while (node != REF_NONE || leaf != REF_NONE) {
        inner_phase<S, COUNT>(A, r, tmin, tmax, node, leaf, st, cnt);
        while (leaf != REF_NONE) {
            if (test_leaf<COUNT>(A, r, tmin, tmax, leaf, skip, true, tb, best, cnt)) return true;
            const bool more = node < 0;
            leaf = more ? node : REF_NONE;
            st.pop(more && node != REF_NONE, tmax, node, leaf);
        }
    }
    return false;
}

// When a packet of rays parts: it has a credit, which a visit changes by the lanes that meet one of the
// node's boxes less 1/4 of all, up to PACKET_CREDIT. The pixels of a pass lie next to one another, but in a
// coarse image of a dense scene, with few samples to a pixel, their rays meet few nodes in common and the
// walk visits what any of them meets: 2M spheres in tight clusters at 320x240, 2 samples, took 2.9 ms
// (2.1 ms lane by lane before the packets), 0.40 ms with the credit; 20M uniform spheres at 800x600, 2
// samples, 0.66 ms and 0.50. Over 480 frames of 12 scenes (10k to 50M spheres, 210x200 to 1886x1060, 2 to
// 64 samples) the mean is 0.80 of the time, and none takes more than 4 % longer. With credits of 256, 1024
// and 4096 the mean is 0.72, 0.76 and 0.85 and the worst 13, 6 and 4 %; with 1/8 of the lanes and 256, 512
// and 1024 0.77, 0.81, 0.85.
constexpr int PACKET_CREDIT = 2048;

// Closest hit of a whole wavefront whose rays lie in one octant of directions, as the samples of a
// pixel do: all lanes walk the same nodes together (a node is visited while any lane's ray meets
// its box before its best hit). The node and its spheres are scalar loads, the stack holds one
// reference with each lane's own entry distance, and since the sign of every direction component
// is the same in all lanes, the near and far planes of a box are picked by scalar selects: a visit
// takes 6 multiply-adds and 5 compares per box, against 6 and 11 lane by lane, and no lane waits
// for another's sphere test. Every lane's result is that of trace_closest. Lanes need not all be
// active (sx, sy, sz: the negative direction components).
// Ends with node REF_NONE or, when its credit is used up, with what each lane goes on from by itself, with
// its own distances on the stack.
template <int S, bool COUNT>
__device__ __forceinline__ void walk_packet(const TraceArgs& A, const RayPre& r, float tmin, float tmax, bool sx, bool sy,
                                            bool sz, int32_t& node_out, int32_t& leaf_out, float& t_best, int& best,
                                            LaneStack<S>& st, Count& cnt) {
    const V3 on = V3{sx ? r.oih.x : r.oil.x, sy ? r.oih.y : r.oil.y, sz ? r.oih.z : r.oil.z};
    const V3 of = V3{sx ? r.oil.x : r.oih.x, sy ? r.oil.y : r.oih.y, sz ? r.oil.z : r.oih.z};
    const int few = (int)__popcll(__ballot(true)) / 4;
    int credit = PACKET_CREDIT;
    int32_t node = 0;
    int sp = 1;
    auto slab_oct = [&](float lx, float ly, float lz, float hx, float hy, float hz) -> float {
        const float xn = __builtin_fmaf(sx ? hx : lx, r.inv.x, -on.x), xf = __builtin_fmaf(sx ? lx : hx, r.inv.x, -of.x);
        const float yn = __builtin_fmaf(sy ? hy : ly, r.inv.y, -on.y), yf = __builtin_fmaf(sy ? ly : hy, r.inv.y, -of.y);
        const float zn = __builtin_fmaf(sz ? hz : lz, r.inv.z, -on.z), zf = __builtin_fmaf(sz ? lz : hz, r.inv.z, -of.z);
        const float tn = fmaxf(fmaxf(xn, yn), fmaxf(zn, tmin));
        const float tf = fminf(fminf(xf, yf), fminf(zf, t_best));
        return tn <= tf ? tn : INFINITY;
    };
    while (node != REF_NONE && credit >= 0) {
        bool pop = true;
        if (node >= 0) {
            const_f32x4 q = (const_f32x4)(uintptr_t)(A.nodes + node);
            const f32x4 a = q[0], b = q[1], c = q[2];
            const i32x4 d = *(const_i32x4)(q + 3);
            if (COUNT) cnt.visits++;
            const float tn0 = slab_oct(a.x, a.y, a.z, a.w, b.x, b.y);
            const float tn1 = slab_oct(b.z, b.w, c.x, c.y, c.z, c.w);
            const uint64_t m0 = __ballot(tn0 != INFINITY), m1 = __ballot(tn1 != INFINITY);
            credit += (int)__popcll(m0 | m1) - few;
            if (m0 && m1) {
                // the child that is nearer for more of the lanes first
                const bool first0 = 2 * __popcll(__ballot(tn0 <= tn1 && tn0 != INFINITY)) >= __popcll(m0 | m1);
                st.sp = sp;
                st.push(true, first0 ? d.y : d.x, first0 ? tn1 : tn0);
                sp = __builtin_amdgcn_readfirstlane(st.sp);
                node = first0 ? d.x : d.y;
                pop = false;
            } else if (m0 | m1) {
                node = m0 ? d.x : d.y;
                pop = false;
            }
        } else {
            const int k0 = ~node;
            const int k1 = (uint32_t)k0 + 1u < A.n_sph ? k0 + 1 : k0;
            if (COUNT) {
                cnt.visits++;
                cnt.pair_visits++;
                cnt.tests += 2;
            }
            const f32x4 v0 = *(const_f32x4)(uintptr_t)(A.leaf_sph + k0), v1 = *(const_f32x4)(uintptr_t)(A.leaf_sph + k1);
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                const f32x4 v = j ? v1 : v0;
                const int leaf = j ? k1 : k0;
                V3 oc;
                float b, e;
                if (!sphere_near(r, make_float4(v.x, v.y, v.z, v.w), oc, b, e)) continue;
                const float t = sphere_far(oc, v.w * v.w, b, e, tmin, tmax);
                if (t >= 0.0f) {
                    if (t < t_best) {
                        t_best = t;
                        best = leaf;
                    } else if (t == t_best && best >= 0 && A.leaf_id[leaf] < A.leaf_id[best]) {
                        best = leaf;
                    }
                }
            }
        }
        if (pop) {  // (at the bottom REF_NONE, nearer than everything)
            i32x2 e;
            do {
                st.sp = sp;
                e = st.take();
                --sp;
            } while (!__ballot(__int_as_float(e.y) <= t_best));
            node = __builtin_amdgcn_readfirstlane(e.x);
            credit = min(credit, PACKET_CREDIT);
        }
    }
    node_out = node;
    st.sp = sp;
    if (node < 0 && node != REF_NONE) {
        leaf_out = node;
        st.pop(true, t_best, node_out, leaf_out);
    }
}

// The closest hit of the active lanes' rays: together where they share an octant of directions and as long
// as they keep together, else lane by lane.
template <int S, bool COUNT>
__device__ __forceinline__ int trace_closest_group(const TraceArgs& A, const RayPre& r, float tmin, float tmax,
                                                   float& t_best, LaneStack<S>& st, Count& cnt) {
    const uint64_t act = __ballot(true);
    const uint64_t bx = __ballot(r.inv.x < 0.0f), by = __ballot(r.inv.y < 0.0f), bz = __ballot(r.inv.z < 0.0f);
    int best = -1;
    t_best = tmax;
    int32_t node = 0, leaf = REF_NONE;
    st.reset();
    if ((bx == 0 || bx == act) && (by == 0 || by == act) && (bz == 0 || bz == act)) {
        walk_packet<S, COUNT>(A, r, tmin, tmax, bx != 0, by != 0, bz != 0, node, leaf, t_best, best, st, cnt);
    } else {
        descend_together<S, COUNT>(A, r, tmin, t_best, node, leaf, st, cnt);
    }
    finish_closest<S, COUNT>(A, r, tmin, tmax, node, leaf, t_best, best, st, cnt);
    return best;
}

// Slab test of one child box returning the entry distance (+inf when missed) and the exit.
__device__ __forceinline__ float slab_io(const RayPre& r, float lx, float ly, float lz, float hx, float hy, float hz,
                                         float tmin, float tmax, float& tf_out) {
    float x0 = __builtin_fmaf(lx, r.inv.x, -r.oil.x), x1 = __builtin_fmaf(hx, r.inv.x, -r.oih.x);
    float y0 = __builtin_fmaf(ly, r.inv.y, -r.oil.y), y1 = __builtin_fmaf(hy, r.inv.y, -r.oih.y);
    float z0 = __builtin_fmaf(lz, r.inv.z, -r.oil.z), z1 = __builtin_fmaf(hz, r.inv.z, -r.oih.z);
    float tn = fmaxf(fmaxf(fminf(x0, x1), fminf(y0, y1)), fmaxf(fminf(z0, z1), tmin));
    float tf = fminf(fminf(fmaxf(x0, x1), fmaxf(y0, y1)), fminf(fmaxf(z0, z1), tmax));
    tf_out = tf;
    return tn <= tf ? tn : INFINITY;
}

// Treelet P-k-d traversal (the interval logic of pkd_intersect, plugins/optix_owl/cuda_resources/
// pkdPrograms.cu:45-159, under a top tree of boxes like the LBVH's). A reference is a top node
// (>= 0) or the P-k-d node at position p (~p): the node's sphere is tested when the ray's
// interval [t0, t1] meets the node's slab (split coordinate -+ the treelet's largest radius,
// widened by the padding every slab test here carries); the near child takes
// [t0, min(slab exit, t1, best)], the far child [max(t0, slab entry), min(t1, best)]. Closed
// intervals, so that equal-t hits still reach the lowest particle id. Before its exact test a
// sphere must also meet the ray in its own box. A pushed P-k-d entry keeps
// its entry distance and resumes with t1 = the best hit at the time it is popped. A treelet is
// entered at its root over its box's [entry, exit].
// The lowest three levels of a treelet are not walked: at a node whose great-grandchildren are past the
// treelet's end the up to 7 spheres of its subtree are fetched together and pass the first part of the
// sphere test (up to its square root) together; the rest runs for the few that pass. Most of the visits
// were there, each a sphere and a split axis behind the one before. As in the LBVH's two phases, a
// wavefront's lanes visit top nodes, then P-k-d nodes, then subtrees, each until at most 3/8 of the lanes
// that began still do: with the two kinds of P-k-d visit in one loop nearly each iteration ran both for
// part of the lanes. 8M clustered spheres at 1280x720, 1-spp AO: 8.1 ms walked to the leaves, 7.3 with
// the lowest two levels together, 6.3 with three, 5.2 with the visits in phases (5.6, 5.2 and 5.3 at 1/8,
// 3/8 and 5/8). At 4, 5, 6 and 7 wavefronts per SIMD 5.5, 5.2, 5.4 and 6.7 (from 6 on it spills). Bound by
// the latency of dependent fetches: the tiles along a line of clusters take nearly the kernel's time.
// Closest hit (ANY false): returns the position of the hit (or -1) and its t in t_best. ANY:
// returns 1 at the first hit of a sphere other than position `skip`, else 0.
template <int S, bool COUNT, bool ANY>
__device__ int trace_tl(const TraceArgs& A, const RayPre& r, float tmin, float tmax, int skip, float& t_best,
                        LaneStack<S>& st, Count& cnt) {
    int best = -1;
    t_best = tmax;
    st.reset();
    int32_t node = 0;
    float t0 = 0.0f, t1 = 0.0f;
    uint32_t cur_tl = 0xffffffffu;
    float rmax = 0.0f;
    const uint32_t lg = A.tl_log2;
    const uint32_t msk = (1u << lg) - 1u;
    auto pop = [&]() {  // (the sentinel ends it)
        i32x2 e;
        do {
            e = st.take();
        } while (__int_as_float(e.y) > t_best);
        node = e.x;
        t0 = __int_as_float(e.y);
        t1 = t_best;
    };
    // whether ref is a P-k-d node above the lowest three levels of its treelet
    auto inner = [&](int32_t ref) -> bool {
        const uint32_t i = ~(uint32_t)ref & msk, bs = ~(uint32_t)ref - i;
        return ref < 0 && ref != REF_NONE && 8 * i + 7 < min(A.n_sph - bs, msk + 1u);
    };
    // a sphere against its own box (centre -+ radius: the leaf box an LBVH traversal tests before
    // its sphere; a filter that changes no result, most spheres near the ray lie off it), then exactly
    auto test = [&](uint32_t p, const float4& sp) -> bool {
        if ((ANY && (int)p == skip) || slab(r, sp.x - sp.w, sp.y - sp.w, sp.z - sp.w, sp.x + sp.w, sp.y + sp.w,
                                            sp.z + sp.w, tmin, t_best) == INFINITY)
            return false;
        if (COUNT) cnt.tests++;
        const float t = sphere_t(r.o, r.d, sp, tmin, tmax);
        if (t >= 0.0f) {
            if (ANY) return true;
            if (t < t_best) {
                t_best = t;
                best = (int)p;
            } else if (t == t_best && best >= 0 && A.leaf_id[p] < A.leaf_id[best]) {
                best = (int)p;
            }
        }
        return false;
    };
    while (node != REF_NONE) {
        const int few_top = (int)__popcll(__ballot(node >= 0)) * 3 / 8;
        while (node >= 0) {
            const float4* q = reinterpret_cast<const float4*>(A.nodes + node);
            const float4 a = q[0], b = q[1], c = q[2];
            const int4 d = reinterpret_cast<const int4*>(q)[3];
            if (COUNT) cnt.visits++;
            float tf0, tf1;
            const float tn0 = slab_io(r, a.x, a.y, a.z, a.w, b.x, b.y, tmin, t_best, tf0);
            const float tn1 = slab_io(r, b.z, b.w, c.x, c.y, c.z, c.w, tmin, t_best, tf1);
            const bool h0 = tn0 != INFINITY && d.x != INT32_MIN, h1 = tn1 != INFINITY && d.y != INT32_MIN;
            // a treelet child ~t becomes the P-k-d root at position t << lg
            const int32_t r0 = d.x >= 0 ? d.x : (int32_t)~((uint32_t)(~d.x) << lg);
            const int32_t r1 = d.y >= 0 ? d.y : (int32_t)~((uint32_t)(~d.y) << lg);
            if (h0 || h1) {
                const bool first0 = h0 && (!h1 || tn0 <= tn1);
                st.push(h0 && h1, first0 ? r1 : r0, first0 ? tn1 : tn0);
                node = first0 ? r0 : r1;
                t0 = first0 ? tn0 : tn1;
                t1 = first0 ? tf0 : tf1;
            } else {
                pop();
            }
            if ((int)__popcll(__ballot(node >= 0)) <= few_top) break;
        }
        // P-k-d nodes down to the lowest three levels
        const int few_in = (int)__popcll(__ballot(inner(node))) * 3 / 8;
        while (inner(node)) {
            const uint32_t p = ~(uint32_t)node;
            const uint32_t tl = p >> lg;
            if (tl != cur_tl) {
                cur_tl = tl;
                rmax = A.tl_rmax[tl];
            }
            const uint32_t i = p & msk, bs = p - i;
            const float4 sp = A.leaf_sph[p];
            const int dd = A.pkd_dim[p];
            if (COUNT) cnt.visits++;
            const float sc = dd == 0 ? sp.x : (dd == 1 ? sp.y : sp.z);
            const float inv = dd == 0 ? r.inv.x : (dd == 1 ? r.inv.y : r.inv.z);
            const float oil = dd == 0 ? r.oil.x : (dd == 1 ? r.oil.y : r.oil.z);
            const float oih = dd == 0 ? r.oih.x : (dd == 1 ? r.oih.y : r.oih.z);
            const float tlo = __builtin_fmaf(sc - rmax, inv, -oil), thi = __builtin_fmaf(sc + rmax, inv, -oih);
            const float tnr = fminf(tlo, thi), tfr = fmaxf(tlo, thi);
            if (fmaxf(t0, tnr) <= fminf(tfr, fminf(t1, t_best)) && test(p, sp)) return 1;  // (true only for ANY)
            const float lim = fminf(t1, t_best);
            const float n_t1 = fminf(tfr, lim), f_t0 = fmaxf(t0, tnr);
            const uint32_t sg = inv < 0.0f ? 1u : 0u;
            const uint32_t nc = 2 * i + 1 + sg, fc = 2 * i + 2 - sg;  // both lie inside the treelet here
            const bool need_n = t0 <= n_t1, need_f = f_t0 <= lim;
            if (need_n) {
                st.push(need_f, ~(int32_t)(bs + fc), f_t0);
                node = ~(int32_t)(bs + nc);
                t1 = n_t1;
            } else if (need_f) {
                node = ~(int32_t)(bs + fc);
                t0 = f_t0;
                t1 = lim;
            } else {
                pop();
            }
            if ((int)__popcll(__ballot(inner(node))) <= few_in) break;
        }
        // the subtrees of the lowest three levels
        const int few_g = (int)__popcll(__ballot(node < 0 && node != REF_NONE && !inner(node))) * 3 / 8;
        while (node < 0 && node != REF_NONE && !inner(node)) {
            const uint32_t p = ~(uint32_t)node;
            const uint32_t i = p & msk, bs = p - i, m = min(A.n_sph - bs, msk + 1u);
            const float4 sp = A.leaf_sph[p];
            // the part of the sphere test before the square root for all seven (a place past the end
            // repeats the node), the rest for the few that pass
            float4 g[6];
#pragma unroll
            for (uint32_t k = 0; k < 6; ++k) {
                const uint32_t c = k < 2 ? 2 * i + 1 + k : 4 * i + 1 + k;
                g[k] = A.leaf_sph[c < m ? bs + c : p];
            }
            if (COUNT) cnt.visits += 7;
            uint32_t near = 0;
#pragma unroll
            for (uint32_t k = 0; k < 7; ++k) {
                V3 oc;
                float b_, e_;
                near |= sphere_near(r, k < 6 ? g[k] : sp, oc, b_, e_) ? 1u << k : 0u;
            }
            bool hit = false;
            while (near) {
                const uint32_t k = __ffs(near) - 1;
                near &= near - 1;
                const uint32_t c = k < 2 ? 2 * i + 1 + k : (k < 6 ? 4 * i + 1 + k : i);
                const uint32_t pc = c < m ? bs + c : p;
                hit = test(pc, A.leaf_sph[pc]);
                if (hit) break;
            }
            if (ANY && hit) return 1;
            pop();
            if ((int)__popcll(__ballot(node < 0 && node != REF_NONE && !inner(node))) <= few_g) break;
        }
    }
    return ANY ? 0 : best;
}

// The structure a kernel traverses: TL = treelet P-k-d trees, else the LBVH.
// TOG: the active lanes' rays are coherent (primary rays).
template <int S, bool COUNT, bool TL, bool TOG>
__device__ __forceinline__ int trace_closest_x(const TraceArgs& A, const RayPre& r, float tmin, float tmax,
                                               float& t_best, LaneStack<S>& st, Count& cnt) {
    if (TL) return trace_tl<S, COUNT, false>(A, r, tmin, tmax, -1, t_best, st, cnt);
    return trace_closest<S, COUNT, TOG>(A, r, tmin, tmax, t_best, st, cnt);
}
template <int S, bool COUNT, bool TL>
__device__ __forceinline__ bool trace_any_x(const TraceArgs& A, const RayPre& r, float tmin, float tmax, int skip,
                                            LaneStack<S>& st, Count& cnt) {
    if (TL) {
        float tb;
        return trace_tl<S, COUNT, true>(A, r, tmin, tmax, skip, tb, st, cnt) != 0;
    }
    return trace_any<S, COUNT>(A, r, tmin, tmax, skip, st, cnt);
}

// Diffuse bounce direction of raygen.cu:71-77,149-152: rejection sample in the unit cube,
// the three draws taken x, y, z in order.
__device__ __forceinline__ V3 random_in_unit_sphere(uint32_t& seed) {
    V3 p;
    do {
        float rx = rnd(seed);
        float ry = rnd(seed);
        float rz = rnd(seed);
        p = V3{2.0f * rx - 1.0f, 2.0f * ry - 1.0f, 2.0f * rz - 1.0f};
    } while (dot(p, p) >= 1.0f);
    return p;
}

// Pixel epilogue of raygen.cu:250-272: average over samples, progressive blend, pseudo depth
// (background on a pixel that no sample hit), then every output buffer.
__device__ __forceinline__ void write_pixel_main(const TraceArgs& A, uint32_t opix, float4 col, float depth,
                                                 float best_t, int best_leaf) {
    const FrameConsts& f = A.fc;
    float fs = (float)f.spp;
    col = make_float4(col.x / fs, col.y / fs, col.z / fs, col.w / fs);
    if (f.accumulate && f.frame_idx > 0) {
        // raygen.cu:254-260, lerp(a, b, t) = a + t * (b - a) (utils_device.h:152-154)
        float4 old = A.out_col[opix];
        float a = 1.0f / (float)(f.frame_idx + 1);
        col = make_float4(old.x + a * (col.x - old.x), old.y + a * (col.y - old.y), old.z + a * (col.z - old.z),
                          old.w + a * (col.w - old.w));
    }
    if (depth < FLT_MAX) {
        depth = (f.depth_c / depth) - f.depth_a;
        depth = 0.5f * (depth + 1.0f);
    } else {
        depth = 1.0f;
        col = make_float4(f.bg[0], f.bg[1], f.bg[2], f.bg[3]);
    }
    A.out_col[opix] = col;
    A.out_depth[opix] = depth;
    A.out_t[opix] = best_t;
    A.out_id[opix] = best_leaf >= 0 ? (int32_t)A.leaf_id[best_leaf] : -1;
    A.out_rgba8[opix] = pack_rgba8(col);
}

// The values are rounded to 32 bits first: without the (empty) statement the compiler may take the
// product or sum that makes one with the conversion as a single operation (v_fma_mixlo_f16), rounded once.
__device__ __forceinline__ uint32_t half2_bits(float lo, float hi) {
    asm("" : "+v"(lo), "+v"(hi));
    return (uint32_t)__half_as_ushort(__float2half(lo)) | ((uint32_t)__half_as_ushort(__float2half(hi)) << 16);
}

// Features of a pixel (8 halves): albedo, normal and t of sample 0's hit (zeros on a miss), then
// the mean AO visibility over the samples.
__device__ __forceinline__ void write_pixel(const TraceArgs& A, uint32_t opix, float4 col, float depth, float best_t,
                                            int best_leaf, float aux[8], float vis_sum) {
    write_pixel_main(A, opix, col, depth, best_t, best_leaf);
    if (A.fc.want_aux) {
        aux[7] = vis_sum / (float)A.fc.spp;
        *reinterpret_cast<uint4*>(A.out_aux + (size_t)opix * 8) = make_uint4(
            half2_bits(aux[0], aux[1]), half2_bits(aux[2], aux[3]), half2_bits(aux[4], aux[5]), half2_bits(aux[6], aux[7]));
    }
}

// The same features written in two parts, so that a kernel need not keep them live over the
// traversal of the remaining samples: halves 0-5 once sample 0's primary ray is resolved, halves
// 6-7 with the pixel.
__device__ __forceinline__ void write_aux_head(const TraceArgs& A, uint32_t opix, float a0, float a1, float a2,
                                               float n0, float n1, float n2) {
    if (A.fc.want_aux) {
        uint3* q = reinterpret_cast<uint3*>(A.out_aux + (size_t)opix * 8);
        *q = make_uint3(half2_bits(a0, a1), half2_bits(a2, n0), half2_bits(n1, n2));
    }
}
__device__ __forceinline__ void write_aux_tail(const TraceArgs& A, uint32_t opix, float t0, float vis_sum) {
    if (A.fc.want_aux)
        *reinterpret_cast<uint32_t*>(A.out_aux + (size_t)opix * 8 + 6) = half2_bits(t0, vis_sum / (float)A.fc.spp);
}

template <int S, int MODE, bool COUNT, bool TL = false>
__device__ void shade_pixel(const TraceArgs& A, uint32_t px, uint32_t py, float pad, LaneStack<S>& st, Count& cnt) {
    const FrameConsts& f = A.fc;
    uint32_t pix = py * f.width + px;  // full-frame index: the random stream of the pixel
    uint32_t opix = (py - f.win_y0) * f.win_w + (px - f.win_x0);  // index in the output window
    uint32_t seed = tea16(pix, f.frame_idx);
    float4 col = make_float4(0.f, 0.f, 0.f, 0.f);
    float depth = FLT_MAX;
    float best_t = INFINITY;
    int best_leaf = -1;
    float aux[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    float vis_sum = 0.0f;
    for (uint32_t s = 0; s < f.spp; ++s) {
        float jx = rnd(seed);
        float jy = rnd(seed);
        V3 o, d;
        primary_ray(f, px, py, jx, jy, o, d);
        RayPre r = prep(o, d, pad);
        float t;
        if (COUNT) cnt.rays++;
        int leaf = trace_closest_x<S, COUNT, TL, true>(A, r, 1e-6f, 1e20f, t, st, cnt);
        float4 sc;
        float ray_depth = FLT_MAX;
        if (leaf < 0) {
            if (MODE == 1)
                sc = make_float4(f.bg[0], f.bg[1], f.bg[2], f.bg[3]);
            else
                sc = make_float4(1.0f * 0.8f, 1.0f * 0.8f, 1.0f * 0.8f, 1.0f);
        } else {
            ray_depth = t;
            float4 sp = A.leaf_sph[leaf];
            uint32_t id = A.leaf_id[leaf];
            V3 P = V3{o.x + t * d.x, o.y + t * d.y, o.z + t * d.z};
            V3 N = V3{P.x - sp.x, P.y - sp.y, P.z - sp.z};
            if (dot(N, d) > 0.0f) N = neg(N);
            N = normalize(N);
            float4 alb = A.col[id];
            if (MODE == 1) {
                uint32_t aseed = tea16(pix, 0xA0000000u + f.frame_idx * 4096u + s);
                V3 ad = ao_direction(N, aseed, s, f.spp);
                RayPre ra = prep(P, ad, pad);
                if (COUNT) cnt.rays++;
                bool occ = trace_any_x<S, COUNT, TL>(A, ra, 0.0f, f.ao_distance, leaf, st, cnt);
                float V = occ ? 0.0f : 1.0f;
                sc = make_float4(alb.x * V, alb.y * V, alb.z * V, 1.0f);
                vis_sum += V;
            } else if (MODE == 2 && f.max_bounces > 0) {
                // raygen.cu:122-155 with maxBounces > 0
                V3 cc = V3{alb.x, alb.y, alb.z};
                V3 ro = o, rd = d;
                float rt = t;
                V3 n = N;
                float4 res;
                for (int dep = 0;; ++dep) {
                    if (dep >= f.max_bounces) {
                        res = make_float4(0.1f, 0.1f, 0.1f, 1.0f);
                        break;
                    }
                    V3 so = V3{ro.x + rt * rd.x, ro.y + rt * rd.y, ro.z + rt * rd.z};
                    V3 ru = random_in_unit_sphere(seed);
                    V3 sd = normalize(V3{n.x + ru.x, n.y + ru.y, n.z + ru.z});
                    RayPre rb = prep(so, sd, pad);
                    float tb;
                    if (COUNT) cnt.rays++;
                    int lb = trace_closest_x<S, COUNT, TL, false>(A, rb, 1e-3f, 1e8f, tb, st, cnt);
                    if (lb < 0) {
                        res = make_float4(cc.x * 0.8f, cc.y * 0.8f, cc.z * 0.8f, 1.0f);
                        break;
                    }
                    float4 sb = A.leaf_sph[lb];
                    float4 ab = A.col[A.leaf_id[lb]];
                    V3 Pb = V3{so.x + tb * sd.x, so.y + tb * sd.y, so.z + tb * sd.z};
                    V3 Nb = V3{Pb.x - sb.x, Pb.y - sb.y, Pb.z - sb.z};
                    if (dot(Nb, sd) > 0.0f) Nb = neg(Nb);
                    n = normalize(Nb);
                    cc = V3{cc.x * ab.x, cc.y * ab.y, cc.z * ab.z};
                    ro = so;
                    rd = sd;
                    rt = tb;
                }
                sc = res;
            } else {
                float sh = 0.2f + 0.6f * fabsf(dot(N, d));
                sc = make_float4(alb.x * sh, alb.y * sh, alb.z * sh, 1.0f);
            }
            if (t < best_t) {
                best_t = t;
                best_leaf = leaf;
            }
            if (s == 0) {
                aux[0] = alb.x; aux[1] = alb.y; aux[2] = alb.z;
                aux[3] = N.x; aux[4] = N.y; aux[5] = N.z;
                aux[6] = t;
            }
        }
        col.x += sc.x;
        col.y += sc.y;
        col.z += sc.z;
        col.w += sc.w;
        depth = fminf(depth, ray_depth);
    }
    write_pixel(A, opix, col, depth, best_t, best_leaf, aux, vis_sum);
}

// Lane per pixel, samples in a loop (every sample count). Held to 72 VGPRs (7 wavefronts per SIMD),
// which the fetch latency needs. With the two-phase traversal a frame of 4-bounce paths (1M spheres,
// 801x600, 1 sample) went from 1.65 to 0.71 ms, with the work queues to 0.61 ms. At 1 sample it now
// beats the refill kernel, which had been the default there (50M spheres, 1080p AO: 0.88 against 0.70
// ms; 60M clustered at 4K: 6.7 against 5.7; 10k spheres at 320x240: 92 against 80 us): bound by the
// vector memory unit's address rate (busy 43-81 % of the time) and by lanes that wait (23-41 % active).
// Small frames (W = 5) are held to 102 VGPRs, with hardly a spill: their wavefronts have one or two tiles
// each and the longest rays are the kernel's time. One sample, W = 5 against 7 at 0.2 to 3.5 tiles per
// wavefront (5 scenes of 100k to 4M spheres, uniform, FCC and clusters; Lambert, AO, 1, 4 and 8 bounces): up to
// 1.5 tiles 0 to 20 % off and at most 2 % longer (as two runs differ), at 1.65 up to 14 % off but 4 bounces over FCC spheres 4 %
// longer, at 1.8 13 % off to 5 % longer, at 1.95 and 2.1 uniform scenes of 1M and more 2 to 23 % longer in
// every mode. So the line is at 1.5, in all modes. It counts the 20 wavefronts a CU holds at W = 5: with
// fewer (blocks_per_cu 2 and 4, mmhrt_render_noalloc) both take the same time within 3 %, or W = 5 up to
// 10 % less.
template <int S, int MODE, bool COUNT, bool STEAL, bool TL = false, int W = TL ? 5 : 7>
__global__ __launch_bounds__(TB) __attribute__((amdgpu_waves_per_eu(W, 8))) void k_trace(TraceArgs A) {
    __shared__ int2 lds_stack[LaneStack<S>::N * TB];
    const uint32_t gtid = blockIdx.x * TB + threadIdx.x;
    LaneStack<S> st(lds_stack + threadIdx.x, A.spill + gtid, A.spill_stride, A.ctr + 1);
    Count cnt;
    // slab padding: a bound on the rounding of the FP32 sphere and slab tests, which scale with
    // the magnitude of ray origins and sphere centres (fc.pad carries max |camera coordinate|)
    const float amax = A.info->absmax;
    const float pad = (fmaxf(A.fc.pad, amax) + amax) * (1.0f / 131072.0f);
    const uint32_t lane = __lane_id();
    const uint32_t gwave = gtid >> 6;
    const uint32_t nwaves = (gridDim.x * TB) >> 6;
    WorkQueue wq(A.ctr, A.n_tiles);
    for (uint32_t it = 0;; ++it) {
        uint32_t tile = STEAL ? wq.grab() : gwave + it * nwaves;
        if (tile >= A.n_tiles) break;
        if (TL && A.order) tile = A.order[wq.rank(tile)];
        uint32_t tx = tile % A.tiles_x, ty = tile / A.tiles_x;
        const uint32_t tw = 1u << A.tw_log2, th = 64u >> A.tw_log2;
        uint32_t px = A.fc.win_x0 + tx * tw + (lane & (tw - 1)), py = A.fc.win_y0 + ty * th + (lane >> A.tw_log2);
        if (px < A.fc.win_x0 + A.fc.win_w && py < A.fc.win_y0 + A.fc.win_h)
            shade_pixel<S, MODE, COUNT, TL>(A, px, py, pad, st, cnt);
    }
    if (COUNT) {
        atomicAdd(reinterpret_cast<unsigned long long*>(A.ctr + 2), (unsigned long long)cnt.visits);
        atomicAdd(reinterpret_cast<unsigned long long*>(A.ctr + 4), (unsigned long long)cnt.tests);
        atomicAdd(reinterpret_cast<unsigned long long*>(A.ctr + 6), (unsigned long long)cnt.rays);
        atomicAdd(reinterpret_cast<unsigned long long*>(A.ctr + 8), (unsigned long long)cnt.pair_visits);
    }
}

// One sample of a Lambert (MODE 0) or AO (MODE 1) pixel, the arithmetic of shade_pixel: the
// sample colour, its depth contribution, the hit (t, leaf), the visibility and, for the
// features, albedo and normal.
template <int S, int MODE, bool COUNT, bool TL = false>
__device__ __forceinline__ void shade_sample(const TraceArgs& A, uint32_t px, uint32_t py, uint32_t pix, uint32_t s,
                                             float jx, float jy, float pad, LaneStack<S>& st, Count& cnt,
                                             float4& sc, float& ray_depth, float& t, int& leaf, float& V,
                                             float4& alb_out, V3& n_out) {
    const FrameConsts& f = A.fc;
    V3 o, d;
    primary_ray(f, px, py, jx, jy, o, d);
    RayPre r = prep(o, d, pad);
    if (COUNT) cnt.rays++;
    if (TL)
        leaf = trace_closest_x<S, COUNT, TL, true>(A, r, 1e-6f, 1e20f, t, st, cnt);
    else
        leaf = trace_closest_group<S, COUNT>(A, r, 1e-6f, 1e20f, t, st, cnt);
    ray_depth = FLT_MAX;
    V = 0.0f;
    if (leaf < 0) {
        if (MODE == 1)
            sc = make_float4(f.bg[0], f.bg[1], f.bg[2], f.bg[3]);
        else
            sc = make_float4(1.0f * 0.8f, 1.0f * 0.8f, 1.0f * 0.8f, 1.0f);
        return;
    }
    ray_depth = t;
    float4 sp = A.leaf_sph[leaf];
    uint32_t id = A.leaf_id[leaf];
    V3 P = V3{o.x + t * d.x, o.y + t * d.y, o.z + t * d.z};
    V3 N = V3{P.x - sp.x, P.y - sp.y, P.z - sp.z};
    if (dot(N, d) > 0.0f) N = neg(N);
    N = normalize(N);
    float4 alb = A.col[id];
    alb_out = alb;
    n_out = N;
    if (MODE == 1) {
        uint32_t aseed = tea16(pix, 0xA0000000u + f.frame_idx * 4096u + s);
        V3 ad = ao_direction(N, aseed, s, f.spp);
        RayPre ra = prep(P, ad, pad);
        if (COUNT) cnt.rays++;
        bool occ = trace_any_x<S, COUNT, TL>(A, ra, 0.0f, f.ao_distance, leaf, st, cnt);
        V = occ ? 0.0f : 1.0f;
        sc = make_float4(alb.x * V, alb.y * V, alb.z * V, 1.0f);
    } else {
        float sh = 0.2f + 0.6f * fabsf(dot(N, d));
        sc = make_float4(alb.x * sh, alb.y * sh, alb.z * sh, 1.0f);
    }
}

// Sample-parallel persistent traversal (MODE 0 Lambert, 1 AO; spp a power of two or a multiple
// of 64). A wavefront takes an 8x8 (tile_w x 64/tile_w) pixel tile and walks it in passes; in a
// pass, the lanes hold L = min(spp, 64) consecutive samples of each of 64/L pixels, so the
// primary rays of a lane group start in one pixel and a background pixel costs one quick pass.
// Sample s of a pixel draws its jitter from the pixel's stream advanced by 2s steps
// (lcg_map), and the group folds its samples into the pixel in sample order (colour sums,
// first strictly nearer hit, visibility, sample-0 features), so every output is bit-identical
// to the lane-per-pixel kernels. The primary rays of a pass begin with one packet walk, the AO rays take the
// two-phase traversal lane by lane; 50M FCC spheres at 1080p, 64-spp AO: 31.5 -> 18.4 ms (bound by
// vector ALU issue before and after; 16 spp of 3M spheres at 1000x621: 3.66 -> 1.97 ms). What a pass
// costs beside its rays was a quarter of the issue: the streams of a unit's pixels are set up together,
// one per lane, four lanes sum a colour component each, the features are written by the lane that has
// them, and a pass without a hit ends there (13.5 -> 12.7 ms, and 1.40 -> 1.34 ms). Held to 72 VGPRs (7
// wavefronts per SIMD, a few registers spilled) like the other lane kernels.
template <int S, int MODE, bool COUNT, bool TL = false>
__global__ __launch_bounds__(TB) __attribute__((amdgpu_waves_per_eu(TL ? 5 : 7, 8))) void k_trace_sl(TraceArgs A) {
    __shared__ int2 lds_stack[LaneStack<S>::N * TB];
    const uint32_t gtid = blockIdx.x * TB + threadIdx.x;
    LaneStack<S> st(lds_stack + threadIdx.x, A.spill + gtid, A.spill_stride, A.ctr + 1);
    Count cnt;
    const FrameConsts& f = A.fc;
    const float amax = A.info->absmax;
    const float pad = (fmaxf(f.pad, amax) + amax) * (1.0f / 131072.0f);
    const uint32_t lane = __lane_id();
    const uint32_t L = f.spp >= 64u ? 64u : f.spp;  // lanes per pixel
    const uint32_t G = 64u / L;                      // pixels per pass
    const uint32_t rounds = f.spp / L;
    const uint32_t g = lane / L, sl = lane % L;
    const uint32_t base = g * L;  // first lane of this lane's pixel group
    const uint32_t tw = 1u << A.tw_log2, th = 64u >> A.tw_log2;
    const uint32_t passes = L >> A.sub_log2;  // of a unit (a tile has 64 / G = L)
    uint32_t ja, jc, ra, rc;  // the random stream's maps over 2 * sl draws and over a round's 2 * L
    lcg_map(2u * sl, ja, jc);
    lcg_map(2u * L, ra, rc);
    WorkQueue wq(A.ctr, A.n_tiles << A.sub_log2);
    for (;;) {
        const uint32_t unit = wq.grab();
        if (unit == 0xffffffffu) break;
        const uint32_t tile = unit >> A.sub_log2, q0 = (unit - (tile << A.sub_log2)) * passes;
        const uint32_t tx = tile % A.tiles_x, ty = tile / A.tiles_x;
        // the stream of the tile's pixel `lane`
        const uint32_t tseed = tea16((f.win_y0 + ty * th + (lane >> A.tw_log2)) * f.width + f.win_x0 + tx * tw +
                                         (lane & (tw - 1)), f.frame_idx);
        for (uint32_t q = q0; q < q0 + passes; ++q) {
            const uint32_t tp = q * G + g;  // pixel of this group inside the tile
            const uint32_t px = f.win_x0 + tx * tw + (tp & (tw - 1)), py = f.win_y0 + ty * th + (tp >> A.tw_log2);
            const bool valid = px < f.win_x0 + f.win_w && py < f.win_y0 + f.win_h;
            const uint32_t pix = py * f.width + px;
            uint32_t seed0 = __shfl(tseed, (int)tp, 64);
            float acc = 0.0f;  // colour sum of component sl
            float4 sc;
            // best_t is the least hit distance over the samples, the pixel's depth (FLT_MAX without a hit)
            float best_t = INFINITY, vis_sum = 0.0f;
            int best_leaf = -1;
            float t0 = 0.0f;  // t of sample 0
            for (uint32_t rd = 0; rd < rounds; ++rd) {
                const uint32_t s = rd * L + sl;
                sc = make_float4(0.f, 0.f, 0.f, 0.f);
                float ray_depth = FLT_MAX, t = INFINITY, V = 0.0f;
                int leaf = -1;
                float4 alb = make_float4(0.f, 0.f, 0.f, 0.f);
                V3 N = V3{0.f, 0.f, 0.f};
                if (valid) {
                    uint32_t seed = ja * seed0 + jc;
                    float jx = rnd(seed);
                    float jy = rnd(seed);
                    shade_sample<S, MODE, COUNT, TL>(A, px, py, pix, s, jx, jy, pad, st, cnt, sc, ray_depth,
                                                            t, leaf, V, alb, N);
                }
                seed0 = ra * seed0 + rc;
                const uint32_t opix = (py - f.win_y0) * f.win_w + (px - f.win_x0);
                if (rd == 0 && valid && sl == 0) {  // features of sample 0
                    write_aux_head(A, opix, alb.x, alb.y, alb.z, N.x, N.y, N.z);
                    if (leaf >= 0) t0 = t;
                }
                // a pixel without a hit takes the background whatever its samples' colours sum to
                if (rounds == 1 && __ballot(leaf >= 0) == 0) break;
                // visibility is 0 or 1 per sample, so its sum is exact in any order: the count of
                // the group's unoccluded hits
                const uint64_t gmask = L == 64u ? ~0ull : ((1ull << L) - 1ull) << base;
                vis_sum += (float)__popcll(__ballot(leaf >= 0 && V > 0.0f) & gmask);
                // the group's closest hit, the first sample of least t (an exchange over lane ^ m
                // stays inside the aligned group of L lanes); an earlier round wins ties
                const float ht = leaf >= 0 ? t : INFINITY;
                float rt = ht;
                for (uint32_t m = L >> 1; m > 0; m >>= 1) rt = fminf(rt, __shfl_xor(rt, (int)m, 64));
                if (rt < best_t) {
                    best_t = rt;
                    best_leaf = __shfl(leaf, __ffsll((unsigned long long)(__ballot(ht == rt) & gmask)) - 1, 64);
                }
                // colours are summed in sample order, a component per lane, through the first two
                // stack rows of the wavefront's lanes (no ray is under way here)
                float* wxy = reinterpret_cast<float*>(lds_stack + (threadIdx.x - lane));
                float* wzw = reinterpret_cast<float*>(lds_stack + TB + (threadIdx.x - lane));
                wxy[lane] = sc.x;
                wxy[64 + lane] = sc.y;
                wzw[lane] = sc.z;
                wzw[64 + lane] = sc.w;
                __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
                __builtin_amdgcn_wave_barrier();
                if (sl < 4u && L > 2u) {
                    const float4* w = reinterpret_cast<const float4*>((sl < 2u ? wxy : wzw) + 64 * (sl & 1u) + base);
                    for (uint32_t i = 0; i < L / 4; ++i) {
                        const float4 v = w[i];
                        acc = acc + v.x + v.y + v.z + v.w;
                    }
                }
                __builtin_amdgcn_wave_barrier();
                __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
            }
            const uint32_t opix = (py - f.win_y0) * f.win_w + (px - f.win_x0);
            float4 col;
            if (L == 2u)  // (0 + sample 0 + sample 1, without the rows)
                col = make_float4(0.0f + sc.x + __shfl(sc.x, (int)base + 1, 64), 0.0f + sc.y + __shfl(sc.y, (int)base + 1, 64),
                                  0.0f + sc.z + __shfl(sc.z, (int)base + 1, 64), 0.0f + sc.w + __shfl(sc.w, (int)base + 1, 64));
            else
                col = make_float4(acc, __shfl(acc, (int)base + 1, 64), __shfl(acc, (int)base + 2, 64),
                                  __shfl(acc, (int)base + 3, 64));
            if (valid && sl == 0) {
                write_pixel_main(A, opix, col, best_t < INFINITY ? best_t : FLT_MAX, best_t, best_leaf);
                write_aux_tail(A, opix, t0, vis_sum);
            }
        }
    }
    if (COUNT) {
        atomicAdd(reinterpret_cast<unsigned long long*>(A.ctr + 2), (unsigned long long)cnt.visits);
        atomicAdd(reinterpret_cast<unsigned long long*>(A.ctr + 4), (unsigned long long)cnt.tests);
        atomicAdd(reinterpret_cast<unsigned long long*>(A.ctr + 6), (unsigned long long)cnt.rays);
        atomicAdd(reinterpret_cast<unsigned long long*>(A.ctr + 8), (unsigned long long)cnt.pair_visits);
    }
}

// Persistent traversal with wavefront-ballot compaction and refill (MODE 0 Lambert, 1 AO).
// Each lane owns one pixel at a time and walks its samples in order (primary ray, then for AO
// one occlusion ray). The inner loop advances every active lane by one node visit and keeps
// going while at least `refill` lanes of the wave still trace; below that the wave leaves the
// loop, finished lanes shade and set up their next ray (next AO ray, next sample, or a new pixel
// taken with one wave-aggregated atomic), and traversal resumes. Per-pixel arithmetic and
// random streams are those of k_trace, so the results are bit-identical.
enum : int { L_IDLE = 0, L_NEED = 1, L_PRIM = 2, L_AO = 3, L_PRIM_DONE = 4, L_AO_DONE = 5, L_OFF = 6 };

// Held to 5 wavefronts per SIMD (at most 102 VGPRs; it takes 96 and spills nothing). Primary and AO
// rays, which a refilled wavefront holds at once, run one instruction stream. Off unless the option
// asks for it (figures at k_trace).
template <int S, int MODE, bool COUNT>
__global__ __launch_bounds__(TB) __attribute__((amdgpu_waves_per_eu(5, 8))) void k_trace_refill(TraceArgs A,
                                                                                                uint32_t refill) {
    __shared__ int2 lds_stack[LaneStack<S>::N * TB];
    const uint32_t gtid = blockIdx.x * TB + threadIdx.x;
    LaneStack<S> st(lds_stack + threadIdx.x, A.spill + gtid, A.spill_stride, A.ctr + 1);
    Count cnt;
    const FrameConsts& f = A.fc;
    const float amax = A.info->absmax;
    const float pad = (fmaxf(f.pad, amax) + amax) * (1.0f / 131072.0f);
    const uint32_t lane = __lane_id();
    const uint32_t tw = 1u << A.tw_log2, th = 64u >> A.tw_log2;
    WorkQueue wq(A.ctr, A.n_tiles);
    uint32_t tile = 0, used = 64u;  // the wavefront's tile and how many of its pixels are taken
    int state = L_IDLE;
    bool exhausted = false;
    // pixel state
    uint32_t px = 0, py = 0, pix = 0, opix = 0, s = 0, seed = 0;
    float4 col = make_float4(0.f, 0.f, 0.f, 0.f);
    // best_t is the least hit distance over the samples, the pixel's depth (FLT_MAX without a hit)
    float best_t = INFINITY, vis_sum = 0.0f;
    int best_leaf_px = -1;
    float aux6 = 0.f;  // t of sample 0's hit (the other features are written when it is found)
    // ray state
    RayPre r;
    float tmin = 0.f, tmax = 0.f, t_best = 0.f;
    int best = -1, skip = -1;
    int32_t node = 0, leaf = REF_NONE;
    float4 alb = make_float4(0.f, 0.f, 0.f, 0.f);
    for (;;) {
        // 1. idle lanes take the next pixels of the wavefront's tile, and of a new one when it is used up
        uint64_t idle = __ballot(state == L_IDLE);
        while (idle && !exhausted) {
            if (used == 64u) {
                tile = wq.grab();
                used = 0;
                if (tile == 0xffffffffu) {
                    exhausted = true;
                    break;
                }
            }
            if (state == L_IDLE) {
                const uint32_t k = used + (uint32_t)__popcll(idle & ((1ull << lane) - 1ull));
                const uint32_t tx = tile % A.tiles_x, ty = tile / A.tiles_x;
                const uint32_t lx = tx * tw + (k & (tw - 1)), ly = ty * th + (k >> A.tw_log2);
                // places past the window edge map to no pixel; the lane simply asks again
                if (k < 64u && lx < f.win_w && ly < f.win_h) {
                    px = f.win_x0 + lx;
                    py = f.win_y0 + ly;
                    pix = py * f.width + px;
                    opix = ly * f.win_w + lx;
                    s = 0;
                    seed = tea16(pix, f.frame_idx);
                    col = make_float4(0.f, 0.f, 0.f, 0.f);
                    best_t = INFINITY;
                    best_leaf_px = -1;
                    vis_sum = 0.0f;
                    aux6 = 0.f;
                    state = L_NEED;
                }
            }
            const uint32_t n = (uint32_t)__popcll(idle);
            used = used + n < 64u ? used + n : 64u;
            idle = __ballot(state == L_IDLE);
        }
        if (exhausted && state == L_IDLE) state = L_OFF;
        // 2. new primary rays
        if (state == L_NEED) {
            float jx = rnd(seed);
            float jy = rnd(seed);
            V3 o, d;
            primary_ray(f, px, py, jx, jy, o, d);
            r = prep(o, d, pad);
            tmin = 1e-6f;
            tmax = 1e20f;
            t_best = tmax;
            best = -1;
            node = 0;
            st.reset();
            if (COUNT) cnt.rays++;
            state = L_PRIM;
        }
        uint64_t act = __ballot(state == L_PRIM || state == L_AO);
        uint64_t live = __ballot(state != L_OFF);
        if (!live) break;
        // 3. traversal: per iteration one inner phase and one leaf phase of the active lanes,
        // primary and AO lanes together (an any-hit ray's bound t_best stays at its tmax)
        while (act) {
            if (state == L_PRIM || state == L_AO) {
                const bool ao = state == L_AO;
                inner_phase<S, COUNT>(A, r, tmin, t_best, node, leaf, st, cnt);
                while (leaf != REF_NONE) {
                    const bool occ = test_leaf<COUNT>(A, r, tmin, tmax, leaf, ao ? skip : -1, ao, t_best, best, cnt);
                    if (occ) {
                        best = 2;
                        node = REF_NONE;
                    }
                    const bool more = node < 0;
                    leaf = more ? node : REF_NONE;
                    st.pop(more && node != REF_NONE, t_best, node, leaf);
                }
                if (node == REF_NONE) state = ao ? L_AO_DONE : L_PRIM_DONE;
            }
            act = __ballot(state == L_PRIM || state == L_AO);
            if ((uint32_t)__popcll(act) < refill) break;
        }
        // 4. shading of finished rays
        bool sample_done = false;
        if (state == L_PRIM_DONE) {
            if (best < 0) {
                float4 sc = MODE == 1 ? make_float4(f.bg[0], f.bg[1], f.bg[2], f.bg[3])
                                      : make_float4(1.0f * 0.8f, 1.0f * 0.8f, 1.0f * 0.8f, 1.0f);
                col.x += sc.x; col.y += sc.y; col.z += sc.z; col.w += sc.w;
                if (s == 0) write_aux_head(A, opix, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f);
                sample_done = true;
            } else {
                float t = t_best;
                float4 sp = A.leaf_sph[best];
                V3 o = r.o, d = r.d;
                V3 Pp = V3{o.x + t * d.x, o.y + t * d.y, o.z + t * d.z};
                V3 N = V3{Pp.x - sp.x, Pp.y - sp.y, Pp.z - sp.z};
                if (dot(N, d) > 0.0f) N = neg(N);
                N = normalize(N);
                alb = A.col[A.leaf_id[best]];
                if (t < best_t) {
                    best_t = t;
                    best_leaf_px = best;
                }
                if (s == 0) {
                    write_aux_head(A, opix, alb.x, alb.y, alb.z, N.x, N.y, N.z);
                    aux6 = t;
                }
                if (MODE == 1) {
                    uint32_t aseed = tea16(pix, 0xA0000000u + f.frame_idx * 4096u + s);
                    V3 ad = ao_direction(N, aseed, s, f.spp);
                    r = prep(Pp, ad, pad);
                    tmin = 0.0f;
                    tmax = f.ao_distance;
                    t_best = tmax;  // an any-hit ray's bound
                    skip = best;
                    best = -1;
                    node = 0;
                    st.reset();
                    if (COUNT) cnt.rays++;
                    state = L_AO;
                } else {
                    float sh = 0.2f + 0.6f * fabsf(dot(N, d));
                    col.x += alb.x * sh; col.y += alb.y * sh; col.z += alb.z * sh; col.w += 1.0f;
                    sample_done = true;
                }
            }
        } else if (state == L_AO_DONE) {
            float V = best == 2 ? 0.0f : 1.0f;
            col.x += alb.x * V; col.y += alb.y * V; col.z += alb.z * V; col.w += 1.0f;
            vis_sum += V;
            sample_done = true;
        }
        if (sample_done) {
            if (++s < f.spp) {
                state = L_NEED;
            } else {
                write_pixel_main(A, opix, col, best_t < INFINITY ? best_t : FLT_MAX, best_t, best_leaf_px);
                write_aux_tail(A, opix, aux6, vis_sum);
                state = L_IDLE;
            }
        }
    }
    if (COUNT) {
        atomicAdd(reinterpret_cast<unsigned long long*>(A.ctr + 2), (unsigned long long)cnt.visits);
        atomicAdd(reinterpret_cast<unsigned long long*>(A.ctr + 4), (unsigned long long)cnt.tests);
        atomicAdd(reinterpret_cast<unsigned long long*>(A.ctr + 6), (unsigned long long)cnt.rays);
        atomicAdd(reinterpret_cast<unsigned long long*>(A.ctr + 8), (unsigned long long)cnt.pair_visits);
    }
}

// Where and how large a trace launch is: at most `blocks` workgroups on a device of `cus` CUs.
struct Grid {
    unsigned blocks, cus;
    hipStream_t stream;
};

// A persistent launch of kernel K, of no more workgroups than are resident at once: a workgroup that
// started only when another had left would find the queues empty but for its wavefronts' own first
// units, and trace those after everything else (1M spheres, 1 sample: 0.48 -> 0.57 ms).
template <auto K, typename... Args>
void launch_resident(const Grid& g, Args... args) {
    static const unsigned per_cu = [] {
        int n = 0;
        if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, K, TB, 0) != hipSuccess || n < 1) {
            (void)hipGetLastError();
            n = 1;
        }
        return (unsigned)n;
    }();
    hipLaunchKernelGGL(K, dim3(std::min(g.blocks, per_cu * g.cus)), dim3(TB), 0, g.stream, args...);
}

template <int S, int MODE, bool COUNT>
void launch3(const TraceArgs& A, const Grid& g, bool steal) {
    if (steal)
        launch_resident<k_trace<S, MODE, COUNT, true>>(g, A);
    else
        launch_resident<k_trace<S, MODE, COUNT, false>>(g, A);
}
template <int S, int MODE>
void launch2(const TraceArgs& A, const Grid& g, bool steal, bool count) {
    if (count)
        launch3<S, MODE, true>(A, g, steal);
    else if (steal && A.fc.spp == 1 && A.n_tiles <= 30 * g.cus)  // 1.5 for each of 20 wavefronts per CU (figures at k_trace)
        launch_resident<k_trace<S, MODE, false, true, false, 5>>(g, A);
    else
        launch3<S, MODE, false>(A, g, steal);
}
template <int S>
void launch1(const TraceArgs& A, const Grid& g, bool steal, bool count, int mode) {
    if (mode == 1)
        launch2<S, 1>(A, g, steal, count);
    else if (mode == 2)
        launch2<S, 2>(A, g, steal, count);
    else
        launch2<S, 0>(A, g, steal, count);
}

template <int S>
void launch_sl(const TraceArgs& A, const Grid& g, bool count, int mode) {
    if (mode == 1) {
        if (count)
            launch_resident<k_trace_sl<S, 1, true>>(g, A);
        else
            launch_resident<k_trace_sl<S, 1, false>>(g, A);
    } else {
        if (count)
            launch_resident<k_trace_sl<S, 0, true>>(g, A);
        else
            launch_resident<k_trace_sl<S, 0, false>>(g, A);
    }
}

// Kernels over the treelet P-k-d trees.
constexpr int TL_STACK = 10 + SPILL_DIST;

// The dearest tiles first. A ray along a line of clusters visits thousands of nodes where the median one
// visits some hundred, one fetch after the other, and a tile of such rays that was begun late ran on by
// itself at the end. The number of treelets whose boxes a tile's middle ray meets tells them apart
// well enough: k_tl_cost counts them in steps of four (one lane per tile, boxes of the top tree only),
// k_tl_order sorts the tiles by it, and the work queues hand out the first tiles of the order before the
// others. 8M clustered spheres at 1280x720: trace 5.2 -> 4.4 ms, for 0.09 ms of counting and 0.015 of
// sorting. For 2 to 8 tiles per wavefront. Ordered against as they lie, Lambert and AO over 6 scenes of 100k
// to 4M spheres: clusters take 3 to 26 % less at every ratio from 1 to 12, most at 2.8 to 4.5. Uniform and
// FCC scenes take up to 14 % longer at 1, 8 % at 1.65, 11 % at 1.8 (AO 9, 7 and 2 %); at 2.05, 2.2 and 2.4
// Lambert frames still take up to 8, 6 and 3 % longer, AO frames 1 % longer to 16 % less; from 2.8 to 9
// nothing takes more than 2 % longer, at 12 AO frames 2 % with half of the gain. Four wavefronts for
// each of the dearest 1/64 to 1/8 of the tiles took 4 to 25 % longer, wavefront priority by age 1 %.
constexpr int TL_TOP = 24;  // stack entries of a walk over the top tree (at most 22 levels)
__global__ __launch_bounds__(TB) void k_tl_cost(TraceArgs A, uint32_t* cost) {
    __shared__ int2 lds_stack[TL_TOP * TB];
    const uint32_t gtid = blockIdx.x * TB + threadIdx.x;
    LaneStack<TL_TOP> st(lds_stack + threadIdx.x, A.spill + gtid, A.spill_stride, A.ctr + 1);
    const FrameConsts& f = A.fc;
    const float amax = A.info->absmax;
    const float pad = (fmaxf(f.pad, amax) + amax) * (1.0f / 131072.0f);
    const uint32_t tw = 1u << A.tw_log2, th = 64u >> A.tw_log2;
    for (uint32_t tile = gtid; tile < A.n_tiles; tile += gridDim.x * TB) {
        const uint32_t tx = tile % A.tiles_x, ty = tile / A.tiles_x;
        const uint32_t px = f.win_x0 + min(tx * tw + tw / 2, f.win_w - 1), py = f.win_y0 + min(ty * th + th / 2, f.win_h - 1);
        V3 o, d;
        primary_ray(f, px, py, 0.5f, 0.5f, o, d);
        const RayPre r = prep(o, d, pad);
        uint32_t met = 0;
        st.reset();
        int32_t node = 0;
        while (node >= 0) {
            const float4* q = reinterpret_cast<const float4*>(A.nodes + node);
            const float4 a = q[0], b = q[1], c = q[2];
            const int2 k = *reinterpret_cast<const int2*>(q + 3);
            const bool h0 = slab(r, a.x, a.y, a.z, a.w, b.x, b.y, 1e-6f, 1e20f) != INFINITY && k.x != INT32_MIN;
            const bool h1 = slab(r, b.z, b.w, c.x, c.y, c.z, c.w, 1e-6f, 1e20f) != INFINITY && k.y != INT32_MIN;
            met += (h0 && k.x < 0) + (h1 && k.y < 0);
            const bool in0 = h0 && k.x >= 0, in1 = h1 && k.y >= 0;
            st.push(in0 && in1, k.y, 0.0f);
            node = in0 ? k.x : (in1 ? k.y : st.take().x);
        }
        cost[tile] = min(met / 4u, 63u);
    }
}
__global__ __launch_bounds__(1024) void k_tl_order(const uint32_t* __restrict__ cost, uint32_t n, uint32_t* order) {
    __shared__ uint32_t bin[64];
    const uint32_t t = threadIdx.x;
    auto each = [&](auto&& body) {  // body(tile, its bin), four tiles' costs fetched at once
        for (uint32_t i0 = t; i0 < n; i0 += 4096) {
            uint32_t c[4];
#pragma unroll
            for (uint32_t k = 0; k < 4; ++k) c[k] = i0 + 1024 * k < n ? cost[i0 + 1024 * k] : 0u;
#pragma unroll
            for (uint32_t k = 0; k < 4; ++k)
                if (i0 + 1024 * k < n) body(i0 + 1024 * k, 63u - c[k]);
        }
    };
    if (t < 64) bin[t] = 0;
    __syncthreads();
    each([&](uint32_t, uint32_t b) { atomicAdd(&bin[b], 1u); });
    __syncthreads();
    if (t < 64) {  // exclusive sums
        const uint32_t v = bin[t];
        uint32_t x = v;
        for (int m = 1; m < 64; m <<= 1) {
            const uint32_t y = __shfl_up(x, m, 64);
            if ((int)t >= m) x += y;
        }
        bin[t] = x - v;
    }
    __syncthreads();
    each([&](uint32_t tile, uint32_t b) { order[atomicAdd(&bin[b], 1u)] = tile; });
}

template <int MODE, bool COUNT>
void launch_tl_m(const TraceArgs& A, const Grid& g, bool sl) {
    if (sl && MODE != 2)
        launch_resident<k_trace_sl<TL_STACK, MODE == 2 ? 0 : MODE, COUNT, true>>(g, A);
    else
        launch_resident<k_trace<TL_STACK, MODE, COUNT, true, true>>(g, A);
}
void launch_tl(const TraceArgs& A, const Grid& g, bool sl, bool count, int mode) {
    if (mode == 1) {
        if (count) launch_tl_m<1, true>(A, g, sl); else launch_tl_m<1, false>(A, g, sl);
    } else if (mode == 2) {
        if (count) launch_tl_m<2, true>(A, g, false); else launch_tl_m<2, false>(A, g, false);
    } else {
        if (count) launch_tl_m<0, true>(A, g, sl); else launch_tl_m<0, false>(A, g, sl);
    }
}

template <int S>
void launch_refill(const TraceArgs& A, const Grid& g, uint32_t refill, bool count, int mode) {
    if (mode == 1) {
        if (count)
            launch_resident<k_trace_refill<S, 1, true>>(g, A, refill);
        else
            launch_resident<k_trace_refill<S, 1, false>>(g, A, refill);
    } else {
        if (count)
            launch_resident<k_trace_refill<S, 0, true>>(g, A, refill);
        else
            launch_resident<k_trace_refill<S, 0, false>>(g, A, refill);
    }
}

// Batched trace: the jobs (timestep, camera) of a series, each with its own timestep's structure
// in its constants, share one persistent launch. The global tile index runs over the concatenated
// tiles of the jobs (prefix[j] = first tile of job j); each wavefront steals tiles and shades them
// with its job's constants and output buffers.
// Held to 72 VGPRs (7 wavefronts per SIMD) like the single-frame kernels.
template <int S, int MODE, bool TL = false>
__global__ __launch_bounds__(TB) __attribute__((amdgpu_waves_per_eu(TL ? 5 : 7, 8))) void k_trace_batch(const TraceArgs* __restrict__ jobs,
                                                    const uint32_t* __restrict__ prefix, uint32_t n_jobs,
                                                    uint32_t* ctr) {
    __shared__ int2 lds_stack[LaneStack<S>::N * TB];
    const uint32_t gtid = blockIdx.x * TB + threadIdx.x;
    LaneStack<S> st(lds_stack + threadIdx.x, jobs[0].spill + gtid, jobs[0].spill_stride, ctr + 1);
    Count cnt;
    const uint32_t lane = __lane_id();
    WorkQueue wq(ctr, prefix[n_jobs]);
    for (;;) {
        const uint32_t tile = wq.grab();
        if (tile == 0xffffffffu) break;
        // the job holding the tile: the last j with prefix[j] <= tile (binary search: a launch
        // over a whole series holds hundreds of jobs)
        uint32_t j = 0, hi = n_jobs - 1;
        while (j < hi) {
            const uint32_t mid = (j + hi + 1) >> 1;
            if (prefix[mid] <= tile)
                j = mid;
            else
                hi = mid - 1;
        }
        const TraceArgs& A = jobs[j];
        const float amax = A.info->absmax;
        const float pad = (fmaxf(A.fc.pad, amax) + amax) * (1.0f / 131072.0f);
        const uint32_t lt = tile - prefix[j];
        const uint32_t tw = 1u << A.tw_log2, th = 64u >> A.tw_log2;
        const uint32_t tx = lt % A.tiles_x, ty = lt / A.tiles_x;
        const uint32_t px = A.fc.win_x0 + tx * tw + (lane & (tw - 1)), py = A.fc.win_y0 + ty * th + (lane >> A.tw_log2);
        if (px < A.fc.win_x0 + A.fc.win_w && py < A.fc.win_y0 + A.fc.win_h)
            shade_pixel<S, MODE, false, TL>(A, px, py, pad, st, cnt);
    }
}

}  // namespace

// One batched launch over jobs that share the mode.
void launch_trace_batch(mmhrt_ctx_s* c, const void* jobs, const uint32_t* prefix, uint32_t n_jobs, uint32_t* ctr,
                        int mode, bool treelets) {
    const Grid g{(unsigned)std::max<int64_t>(1, c->cu_count * c->opt_blocks_per_cu), (unsigned)c->cu_count, c->stream};
    const TraceArgs* J = static_cast<const TraceArgs*>(jobs);
    int S = (int)c->opt_stack_lds;
    launch_fill_u32(c->stream, ctr, 0u, TRACE_CTR_WORDS);
    if (treelets) {  // treelet P-k-d trees
        if (mode == 1)
            launch_resident<k_trace_batch<TL_STACK, 1, true>>(g, J, prefix, n_jobs, ctr);
        else
            launch_resident<k_trace_batch<TL_STACK, 0, true>>(g, J, prefix, n_jobs, ctr);
        return;
    }
#define MMHRT_BATCH(SV)                                                     \
    if (mode == 1)                                                          \
        launch_resident<k_trace_batch<SV, 1>>(g, J, prefix, n_jobs, ctr);   \
    else                                                                    \
        launch_resident<k_trace_batch<SV, 0>>(g, J, prefix, n_jobs, ctr);
    switch (S) {
    case 8: MMHRT_BATCH(6) break;
    case 24: MMHRT_BATCH(14) break;
    case 32: MMHRT_BATCH(18) break;
    default: MMHRT_BATCH(10) break;
    }
#undef MMHRT_BATCH
}

// Job constants for the batched kernel, written into a host buffer of batch_job_size() bytes.
size_t batch_job_size() { return sizeof(TraceArgs); }
int batch_fill_job(mmhrt_ctx_s* c, const FrameConsts& fc, size_t out_offset, void* dst) {
    uint32_t W = fc.win_w, H = fc.win_h;
    (void)H;
    TraceArgs A;
    A.nodes = c->nodes.p;
    A.leaf_sph = c->leaf_sph.p;
    A.leaf_id = c->leaf_id.p;
    A.col = c->ts_col.p;  // the timesteps' own colours, not the context's
    A.info = c->info.p;
    A.spill = c->spill.p;
    A.spill_stride = (uint32_t)(std::max<int64_t>(1, c->cu_count * c->opt_blocks_per_cu) * TB);
    A.ctr = nullptr;
    A.tw_log2 = tile_log2(c->opt_tile_w);
    A.tiles_x = (W + (1u << A.tw_log2) - 1) >> A.tw_log2;
    A.n_tiles = A.tiles_x * ((fc.win_h + (64u >> A.tw_log2) - 1) / (64u >> A.tw_log2));
    A.out_col = c->bt_col.p + out_offset;
    A.out_depth = c->bt_depth.p + out_offset;
    A.out_t = c->bt_t.p + out_offset;
    A.out_id = c->bt_id.p + out_offset;
    A.out_rgba8 = c->bt_rgba8.p + out_offset;
    A.out_aux = nullptr;
    A.pkd_dim = c->accel == 1 ? c->pkd_dim.p : nullptr;
    A.tl_rmax = c->accel == 1 ? c->tl_rmax.p : nullptr;
    A.n_sph = (uint32_t)c->n;
    A.tl_log2 = 0;
    while ((1u << A.tl_log2) < c->pkd_M) ++A.tl_log2;
    A.sub_log2 = 0;
    A.order = nullptr;
    A.fc = fc;
    A.fc.want_aux = 0;
    A.fc.accumulate = 0;
    std::memcpy(dst, &A, sizeof A);
    return (int)A.n_tiles;
}

// tile width option -> log2 (1, 2, 4, 8, 16, 32 or 64 pixels wide; 64 pixels per tile)
uint32_t tile_log2(int64_t tw) {
    uint32_t l = 3;
    for (uint32_t k = 0; k <= 6; ++k)
        if ((int64_t)(1u << k) == tw) l = k;
    return l;
}

namespace {
// Units of work the sample-lanes kernel wants per wavefront. 64-spp AO of 50M spheres at 1080p: 18.4 ms
// in whole tiles, 15.4, 14.4, 13.8 and 13.8 ms at 4, 8, 16 and 32: the last tiles of 64 passes each ran
// on an idle device. Units of fewer than four passes only up to FEW_UNITS: a unit's random streams are
// set up together (16 spp of 3M spheres at 1000x621: 1.42 ms at one pass per unit, 1.34 at four; 800x600
// at 8 spp, 1M spheres: 0.72 ms so, 0.78 and 0.90 with FEW_UNITS 2 and 1).
constexpr uint64_t SUB_UNITS = 16, FEW_UNITS = 4;

// Kernel choice for one frame (the same for both entry points): sample-parallel lanes for Lambert
// and AO with spp a power of two up to 64 or a multiple of 64, the ballot-refill kernel when a
// refill threshold is set, else the lane-per-pixel kernel.
void dispatch_trace(mmhrt_ctx_s* c, TraceArgs& A, unsigned grid, bool count, uint32_t* order) {
    const FrameConsts& fc = A.fc;
    int S = (int)c->opt_stack_lds;
    if (S != 8 && S != 16 && S != 24 && S != 32) S = 16;
    bool steal = c->opt_persistent != 0;
    const int64_t rq = c->opt_refill;
    uint32_t refill = (uint32_t)std::max<int64_t>(0, std::min<int64_t>(64, rq));
    const bool sl_shape = fc.spp > 1 && ((fc.spp >= 64 && fc.spp % 64 == 0) || (fc.spp < 64 && 64 % fc.spp == 0));
    const bool sl = c->opt_sample_lanes != 0 && fc.mode != 2 && sl_shape && (c->accel == 1 || refill == 0);
    // the sample-lanes kernel divides its tiles (min(spp, 64) passes each) until every wavefront
    // of the full grid has its units, and no launch has more wavefronts than units
    if (sl)
        for (uint32_t p = std::min(fc.spp, 64u);
             p > 1 && ((uint64_t)A.n_tiles << A.sub_log2) < (p > 4 ? SUB_UNITS : FEW_UNITS) * grid * (TB / 64); p >>= 1)
            ++A.sub_log2;
    const uint64_t need = (((uint64_t)A.n_tiles << A.sub_log2) + TB / 64 - 1) / (TB / 64);
    const Grid g{(unsigned)std::min<uint64_t>(grid, need), (unsigned)c->cu_count, c->stream};
    if (c->accel == 1) {
        // treelet P-k-d trees: the sample-lanes kernel where the samples fill the lanes, else
        // lane per pixel with work stealing, the dearest tiles first
        const uint32_t waves = 5 * 4 * (uint32_t)c->cu_count;  // at once
        if (!sl && order && A.n_tiles > 2 * waves && A.n_tiles <= 8 * waves) {
            const unsigned blocks = std::min<unsigned>((A.n_tiles + TB - 1) / TB, grid);
            hipLaunchKernelGGL(k_tl_cost, dim3(blocks), dim3(TB), 0, c->stream, A, order);
            hipLaunchKernelGGL(k_tl_order, dim3(1), dim3(1024), 0, c->stream, order, A.n_tiles, order + A.n_tiles);
            A.order = order + A.n_tiles;
        }
        launch_tl(A, g, sl, count, fc.mode);
        return;
    }
    if (sl) {
        switch (S) {
        case 8: launch_sl<6>(A, g, count, fc.mode); break;
        case 24: launch_sl<14>(A, g, count, fc.mode); break;
        case 32: launch_sl<18>(A, g, count, fc.mode); break;
        default: launch_sl<10>(A, g, count, fc.mode); break;
        }
    } else if (refill > 0 && fc.mode != 2) {
        switch (S) {
        case 8: launch_refill<6>(A, g, refill, count, fc.mode); break;
        case 24: launch_refill<14>(A, g, refill, count, fc.mode); break;
        case 32: launch_refill<18>(A, g, refill, count, fc.mode); break;
        default: launch_refill<10>(A, g, refill, count, fc.mode); break;
        }
    } else {
        switch (S) {
        case 8: launch1<6>(A, g, steal, count, fc.mode); break;
        case 24: launch1<14>(A, g, steal, count, fc.mode); break;
        case 32: launch1<18>(A, g, steal, count, fc.mode); break;
        default: launch1<10>(A, g, steal, count, fc.mode); break;
        }
    }
}

void fill_scene_args(mmhrt_ctx_s* c, const FrameConsts& fc, TraceArgs& A) {
    A.nodes = c->nodes.p;
    A.leaf_sph = c->leaf_sph.p;
    A.leaf_id = c->leaf_id.p;
    A.col = c->col.p;
    A.info = c->info.p;
    A.pkd_dim = c->accel == 1 ? c->pkd_dim.p : nullptr;
    A.tl_rmax = c->accel == 1 ? c->tl_rmax.p : nullptr;
    A.n_sph = (uint32_t)c->n;
    uint32_t lg = 0;
    while ((1u << lg) < c->pkd_M) ++lg;
    A.tl_log2 = lg;
    A.tw_log2 = tile_log2(c->opt_tile_w);
    A.tiles_x = (fc.win_w + (1u << A.tw_log2) - 1) >> A.tw_log2;
    A.n_tiles = A.tiles_x * ((fc.win_h + (64u >> A.tw_log2) - 1) / (64u >> A.tw_log2));
    A.sub_log2 = 0;
    A.order = nullptr;
    A.fc = fc;
}

}  // namespace

int render_frame(mmhrt_ctx_s* c, const FrameConsts& fc) {
    uint32_t W = fc.win_w, H = fc.win_h;  // output size = the rendered window
    size_t P = (size_t)W * H;
    int e = 0;
    if ((e = ensure(c, c->fb_col, P, "framebuffer colour"))) return e;
    if ((e = ensure(c, c->fb_depth, P, "framebuffer depth"))) return e;
    if ((e = ensure(c, c->fb_t, P, "framebuffer t"))) return e;
    if ((e = ensure(c, c->fb_id, P, "framebuffer id"))) return e;
    if ((e = ensure(c, c->fb_rgba8, P, "framebuffer rgba8"))) return e;
    if (fc.want_aux && (e = ensure(c, c->fb_aux, P * 8, "framebuffer aux"))) return e;
    if ((e = ensure(c, c->counters, TRACE_CTR_WORDS, "counters"))) return e;
    unsigned grid = (unsigned)(c->cu_count * c->opt_blocks_per_cu);
    if (grid == 0) grid = 1;
    uint32_t lanes = grid * TB;
    if ((e = ensure(c, c->spill, (size_t)lanes * TRACE_SPILL_PER_LANE, "traversal spill"))) return e;
    c->fb_w = W;
    c->fb_h = H;
    c->fb_x0 = fc.win_x0;
    c->fb_y0 = fc.win_y0;
    c->fb_full_w = fc.width;
    c->fb_full_h = fc.height;
    FrameOutputs out{c->fb_col.p, c->fb_depth.p, c->fb_t.p, c->fb_id.p, c->fb_rgba8.p,
                     fc.want_aux ? c->fb_aux.p : nullptr};
    uint32_t* order = nullptr;  // treelets: two words per tile (of at least 64 pixels of the padded window)
    if (c->accel == 1) {
        const uint32_t tw = 1u << tile_log2(c->opt_tile_w), th = 64u / tw;
        if ((e = ensure(c, c->tile_order, 2 * (size_t)((W + tw - 1) / tw) * ((H + th - 1) / th), "tile order"))) return e;
        order = c->tile_order.p;
    }
    return render_frame_into(c, fc, out, c->counters.p, c->spill.p, lanes, c->opt_count != 0, order);
}

// The frame into the given device outputs: the persistent grid is capped at `lanes`, whose
// traversal stacks spill into `spill` (lanes x TRACE_SPILL_PER_LANE words, lane-interleaved);
// `ctr` (TRACE_CTR_WORDS words) takes the overflow flag, the instrumentation counters and the work queues'
// counters and is cleared here by a fill kernel (safe under graph capture). `order` (two words per
// tile, or null) takes the order of a treelet frame's tiles. Allocates nothing.
int render_frame_into(mmhrt_ctx_s* c, const FrameConsts& fc, const FrameOutputs& out, uint32_t* ctr, int32_t* spill,
                      uint32_t lanes, bool count, uint32_t* order) {
    unsigned grid = (unsigned)std::max<int64_t>(1, std::min<int64_t>(c->cu_count * c->opt_blocks_per_cu, lanes / TB));
    TraceArgs A;
    fill_scene_args(c, fc, A);
    A.ctr = ctr;
    A.spill = spill;
    A.spill_stride = grid * TB;
    A.out_col = out.color;
    A.out_depth = out.depth;
    A.out_t = out.t;
    A.out_id = out.hit_id;
    A.out_rgba8 = out.rgba8;
    A.out_aux = fc.want_aux ? out.aux : nullptr;
    launch_fill_u32(c->stream, ctr, 0u, TRACE_CTR_WORDS);
    rec(c, 6);
    dispatch_trace(c, A, grid, count, order);
    rec(c, 7);
    hipError_t he = hipGetLastError();
    if (he != hipSuccess) return hip_fail(c, he, "trace launch");
    return 0;
}

}  // namespace mmhrt
