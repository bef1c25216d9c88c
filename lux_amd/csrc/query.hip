// query.hip -- closest-hit, any-hit and AABB-overlap queries over the
// right-first preorder stackless LBVH. Closest and any hit take the
// near-child-first walk over four-child records (wide.hpp), which returns what
// the preorder walk below returns; rays that it cannot settle take that walk.
//
// Preorder walk rule (src/bvh/bvh_device.cuh:59-87): test node i; on a miss or after a
// leaf jump to nodes[i].escape, on an internal hit step to i+1. With the nodes in
// right-first preorder this visits nodes in the pop order of the host stack
// traversal (src/bvh/cpu_bvh_traversal.h:37-78), so the shrinking t_max and the
// winner of exact-t ties are those of the host LBVH.
//
// Each walk also checks that it moves forward (escape and i+1 are always greater
// than i in preorder), so a damaged node array ends the walk instead of looping.
#include <algorithm>

#include "lux_runtime.hpp"
#include "wide.hpp"

namespace lux {
namespace {

// 64 threads (one wave) per block for the ray queries: a workgroup's resources
// are freed only when its last wave ends, so a finished wave's slot would wait
// for its siblings (the gathered two-child walks measured 822 Mrays/s at 64, 802
// at 128 and 791 at 256). The LDS stack is 5 KiB per block.
constexpr int kBlock = 64;
// The plain copy: 128-thread blocks, at most 4096 of them (4.8 TB/s on 1 GiB;
// other shapes from 2048 to 16384 blocks of 256 or 512 threads measured
// 4.3-5.0 TB/s).
constexpr int kCopyBlock = 128;

struct RayIn {
    f3 o, d;
    float t_min, t_max;
};

__device__ __forceinline__ RayIn load_ray(const lux_ray* rays, int i) {
    const float* p = reinterpret_cast<const float*>(rays + i);
    RayIn r;
    r.o = make3(p[0], p[1], p[2]);
    r.d = make3(p[3], p[4], p[5]);
    r.t_min = p[6];
    r.t_max = p[7];
    return r;
}

__device__ __forceinline__ void load_tri(const lux_triangle* tris, int i, f3& v0, f3& v1, f3& v2) {
    const float* p = reinterpret_cast<const float*>(tris + i);
    v0 = make3(p[0], p[1], p[2]);
    v1 = make3(p[3], p[4], p[5]);
    v2 = make3(p[6], p[7], p[8]);
}

// The tree as the ray kernels read it: the right-first preorder node array and
// the four-child records over it (wide.hpp).
struct RayTree {
    const lux_bvh_node* nodes;
    const WideNode* wide;
    const int32_t* wide_leaf;
    int node_count;    // 2 n - 1
    uint32_t records;  // n - 1, or 0: the preorder walk only
};

// Right-first preorder walk: the rays that the wide walk hands back, one-leaf
// trees and trees beyond 32-bit record offsets.
// kAny = false: closest hit; kAny = true: stop at the first accepted triangle.
// visits/tests count node loads and triangle tests (only read by the stats kernel).
template <bool kAny>
__device__ __forceinline__ int walk_preorder(const lux_bvh_node* __restrict__ nodes, int node_count,
                                          const lux_triangle* __restrict__ tris, int tri_count, const RayIn& ray,
                                          float& t_best, DevInfo* info, uint32_t& visits, uint32_t& tests) {
    const SlabRay sr = make_slab_ray(ray.o, ray.d, ray.t_min);
    float t_max = __builtin_canonicalizef(ray.t_max);
    int best = -1;
    int k = 0;
    bool bad_prim = false, bad_order = false;
    while (uint32_t(k) < uint32_t(node_count)) {
        float4 a, b;
        load_node(nodes, k, a, b);
        ++visits;
        const int prim = __float_as_int(b.z);
        const bool pass = slab_hit(sr, t_max, a.x, a.y, a.z, a.w, b.x, b.y);
        int next = (pass && prim < 0) ? k + 1 : __float_as_int(b.w);
        bad_prim |= pass && prim >= tri_count;
        if (pass && prim >= 0 && prim < tri_count) {
            f3 v0, v1, v2;
            load_tri(tris, prim, v0, v1, v2);
            ++tests;
            float t, u, v;
            if (tri_hit(ray.o, ray.d, ray.t_min, t_max, v0, v1, v2, t, u, v)) {
                best = prim;
                t_max = t;
                if (kAny) next = -1;  // done
            }
        }
        if (next >= 0 && next <= k) {  // preorder positions only grow
            bad_order = true;
            break;
        }
        k = next;
    }
    if (bad_prim) set_error(info, kErrPrimRange);
    if (bad_order) set_error(info, kErrWalkOrder);
    t_best = t_max;
    return best;
}

// What one lane's walk of a ray found: a hit's primitive (-1: none), its leaf
// child (4 * record + child) and distance (a miss: the ray's t_max), and whether
// the ray is the preorder walk's to decide.
struct Found {
    int best = -1;
    uint32_t at = 0;
    float t = 0;
    bool failed = false;
};

// A lane's walk (wide.hpp) of the boxes met in [lo, hi] of its ray; sr.t_min =
// lo. `group` lanes in a row (a power of two) walk one ray between them and share
// the nearest hit (any hit: that there is one); with `skip` a lane only listens.
template <bool kAny>
__device__ __forceinline__ Found walk_part(const RayTree& tree, const lux_triangle* __restrict__ tris, int tri_count,
                                           const RayIn& ray, const SlabRay& sr, float hi, int group, bool skip, uint32_t* stack,
                                           DevInfo* info, uint32_t& visits, uint32_t& tests) {
    Found f;
    f.t = __builtin_canonicalizef(ray.t_max);
    float t_cull = wide_bound(hi);
    bool bad = false, bad_prim = false;
    auto leaf = [&](uint32_t at, uint32_t ref) {
        const uint32_t prim = ref & kIndexMask;
        if (prim >= uint32_t(tri_count)) {
            bad_prim |= ref != kWideEmpty;
            return false;
        }
        f3 v0, v1, v2;
        load_tri(tris, int(prim), v0, v1, v2);
        ++tests;
        float t, u, v;
        if (!tri_uvt(ray.o, ray.d, v0, v1, v2, t, u, v) || !(t > ray.t_min)) return false;
        if (t < f.t || (!kAny && f.best >= 0 && t == f.t && tree.wide_leaf[at] < tree.wide_leaf[f.at])) {
            f.best = int(prim);
            f.at = at;
            if (kAny) return true;
            f.t = t;
            t_cull = fminf(t_cull, t + fabsf(t) * kSoftWindow);
        }
        return false;
    };
    auto share = [&]() {
        if (group == 1) return false;
        if (kAny) {
            int any = f.best >= 0;
            for (int off = 1; off < group; off <<= 1) any |= __shfl_xor(any, off, 64);
            return any != 0;
        }
        float t = f.best >= 0 ? f.t : INFINITY;
        for (int off = 1; off < group; off <<= 1) t = fminf(t, __shfl_xor(t, off, 64));
        t_cull = fminf(t_cull, t + fabsf(t) * kSoftWindow);
        return false;
    };
    const bool done =
        wave_any_parallel(sr)
            ? wide_walk<true>(tree.wide, tree.records, sr, t_cull, skip, stack, kBlock, visits, bad, leaf, share)
            : wide_walk<false>(tree.wide, tree.records, sr, t_cull, skip, stack, kBlock, visits, bad, leaf, share);
    if (bad_prim) set_error(info, kErrPrimRange);
    if (bad) set_error(info, kErrWalkOrder);
    f.failed = !done;
    return f;
}

// One ray on one lane. A ray the wide walk cannot settle is walked again in
// preorder. With t_max fixed, whether a leaf's box passes does not depend on the
// visit order, so an any-hit walk may end at any triangle hit in a leaf whose own
// box passes; near child first meets one soon.
template <bool kAny>
__device__ __forceinline__ int trace_one(const RayTree& tree, const lux_triangle* __restrict__ tris, int tri_count,
                                         const RayIn& ray, float& t_best, uint32_t* stack, DevInfo* info,
                                         uint32_t& visits, uint32_t& tests) {
    if (tree.records != 0 && wide_takes(ray.d)) {
        const SlabRay sr = make_slab_ray(ray.o, ray.d, ray.t_min);
        const Found f =
            walk_part<kAny>(tree, tris, tri_count, ray, sr, ray.t_max, 1, false, stack, info, visits, tests);
        if (!f.failed && (f.best < 0 || wide_settled(tree.nodes, tree.wide_leaf[f.at], sr, f.t))) {
            t_best = f.t;
            return f.best;
        }
    }
    return walk_preorder<kAny>(tree.nodes, tree.node_count, tris, tri_count, ray, t_best, info, visits, tests);
}

template <bool kAny>
__device__ __forceinline__ void store_result(void* __restrict__ out, int ray, int id, float t) {
    if (kAny) {
        static_cast<uint8_t*>(out)[ray] = id >= 0 ? 1 : 0;
    } else {
        lux_hit h;
        h.primitive_id = id;
        h.t = id >= 0 ? t : INFINITY;
        static_cast<lux_hit*>(out)[ray] = h;
    }
}

// One ray per lane in `order` (a permutation of [0, n), or input order); the
// result lands at the ray's own index: a lux_hit, or one byte (kAny).
// Bound by VALU issue (154 instructions a step, 26 % of the lanes busy, since a
// wave lasts as long as its longest walk) with the texture path close behind (data
// return 88 % busy). On 2^22 random rays through 2^20 random triangles: 4.41 ms
// over sibling pairs (386 steps for a wave's longest ray), 3.2 ms over records
// (192 steps). 8 waves a SIMD (64 VGPRs, 12 bytes spilled) take 3.24 ms with the
// sort, 70 VGPRs at 7 waves 3.39 ms. Lanes refilled with new rays as theirs end
// (from runs of 128 to 512 rays a wave, or from one pool per XCD) took 3.5 to
// 5.2 ms: they keep more lanes busy but the wave's rays drift apart in the tree,
// and the loads miss L1. Stack entries that carry their box's entry, to drop them
// when a nearer hit is held, need 6 KiB a wave and took 4.3 ms.
template <bool kAny>
__global__ __launch_bounds__(kBlock) __attribute__((amdgpu_waves_per_eu(8))) void k_trace(
    RayTree tree, const lux_triangle* __restrict__ tris, int tri_count, const lux_ray* __restrict__ rays, int n,
    const uint32_t* __restrict__ order, void* __restrict__ out, DevInfo* info) {
    __shared__ uint32_t stack[kWideStack * kBlock];
    const int i = int(xcd_block()) * kBlock + threadIdx.x;
    if (i >= n) return;
    const int ray = order ? int(order[i]) : i;
    if (uint32_t(ray) >= uint32_t(n)) {  // only if the sort itself reported an error
        set_error(info, kErrSpinLimit);
        return;
    }
    const RayIn r = load_ray(rays, ray);
    float t;
    uint32_t visits = 0, tests = 0;
    const int id = trace_one<kAny>(tree, tris, tri_count, r, t, stack + threadIdx.x, info, visits, tests);
    store_result<kAny>(out, ray, id, t);
}

// Few rays: `group` lanes (a power of two up to 64) walk one ray, each a part of
// the interval in which it meets the root box. A call that leaves most of the
// chip idle lasts as long as its longest walk, a chain of dependent loads; parts
// cut the chain (2^20 random triangles, 2^14 random rays: 330 records for the
// longest ray, 148 in 4 parts, 87 in 8) for more records in all (50, 130 and 194
// a ray). A box met by the ray in [t_min, t_max] is met in some part, so every
// triangle the whole walk tests is tested by some lane; the hit is the smallest
// (t, preorder position) over the lanes, as it is over one lane's walk.
template <bool kAny>
__global__ __launch_bounds__(kBlock) void k_trace_parts(RayTree tree, const lux_triangle* __restrict__ tris,
                                                        int tri_count, const lux_ray* __restrict__ rays, int n,
                                                        const uint32_t* __restrict__ order, int group,
                                                        void* __restrict__ out, DevInfo* info) {
    __shared__ uint32_t stack[kWideStack * kBlock];
    const int i = (int(xcd_block()) * kBlock + int(threadIdx.x)) / group;
    if (i >= n) return;  // whole groups
    const int part = int(threadIdx.x) & (group - 1);
    const int ray = order ? int(order[i]) : i;
    if (uint32_t(ray) >= uint32_t(n)) {
        set_error(info, kErrSpinLimit);
        return;
    }
    const RayIn r = load_ray(rays, ray);
    uint32_t visits = 0, tests = 0;
    int id = -1;
    float t = 0;
    bool settled = false;
    if (wide_takes(r.d)) {  // the same on every lane of the group
        SlabRay sr = make_slab_ray(r.o, r.d, r.t_min);
        // the root box, with a margin; an interval that is empty or not finite
        // leaves the whole ray to the first lane
        float4 a, b;
        load_node(tree.nodes, 0, a, b);
        float enter;
        (void)slab_near<true>(sr, INFINITY, a.x, a.y, a.z, a.w, b.x, b.y, enter);
        const float fx = (sr.neg_x ? a.x : a.w) - r.o.x, fy = (sr.neg_y ? a.y : b.x) - r.o.y,
                    fz = (sr.neg_z ? a.z : b.y) - r.o.z;
        float leave = r.t_max;
        if (!sr.par_x) leave = fminf(leave, fx * sr.inv.x);
        if (!sr.par_y) leave = fminf(leave, fy * sr.inv.y);
        if (!sr.par_z) leave = fminf(leave, fz * sr.inv.z);
        const float step = (leave - enter) / float(group);
        const bool cut = step > 0.0f && step < 1e30f;
        const float lo = enter + step * float(part), hi = enter + step * float(part + 1);
        if (cut && part != 0) sr.t_min = lo;
        const Found f = walk_part<kAny>(tree, tris, tri_count, r, sr, cut && part + 1 < group ? hi : r.t_max, group,
                                        !cut && part != 0, stack + threadIdx.x, info, visits, tests);
        sr.t_min = r.t_min;
        // the smallest (t, position) of the group, on every lane
        int pos = f.best >= 0 ? tree.wide_leaf[f.at] : INT32_MAX;
        float bt = f.best >= 0 ? f.t : INFINITY;
        int bid = f.best, fail = f.failed;
        for (int off = 1; off < group; off <<= 1) {
            const float ot = __shfl_xor(bt, off, 64);
            const int op = __shfl_xor(pos, off, 64), oid = __shfl_xor(bid, off, 64);
            fail |= __shfl_xor(fail, off, 64);
            if (oid >= 0 && (bid < 0 || (kAny ? op < pos : (ot < bt || (ot == bt && op < pos))))) {
                bt = ot;
                pos = op;
                bid = oid;
            }
        }
        id = bid;
        t = bt;
        settled = !fail && (bid < 0 || wide_settled(tree.nodes, pos, sr, kAny ? r.t_max : bt));
    }
    if (part != 0) return;
    if (!settled) id = walk_preorder<kAny>(tree.nodes, tree.node_count, tris, tri_count, r, t, info, visits, tests);
    store_result<kAny>(out, ray, id, t);
}

// The walks of the handle, counting per ray the 32-byte node units loaded (two
// a record) and the triangle tests (summed per wave, one atomic per wave):
// stats[0..2] closest-hit {nodes, 0, tests}, stats[3..5] any-hit {nodes, 0,
// tests}. Rays handed to the preorder walk count both walks. Used to state the
// bytes a traversal actually touches.
__global__ __launch_bounds__(kBlock) void k_trace_stats(RayTree tree, const lux_triangle* __restrict__ tris,
                                                        int tri_count, const lux_ray* __restrict__ rays, int n,
                                                        unsigned long long* stats, DevInfo* info) {
    __shared__ uint32_t stack[kWideStack * kBlock];
    int i = blockIdx.x * kBlock + threadIdx.x;
    uint32_t v0 = 0, t0 = 0, v1 = 0, t1 = 0;
    if (i < n) {
        RayIn r = load_ray(rays, i);
        float t;
        trace_one<false>(tree, tris, tri_count, r, t, stack + threadIdx.x, info, v0, t0);
        trace_one<true>(tree, tris, tri_count, r, t, stack + threadIdx.x, info, v1, t1);
    }
    unsigned long long c[6] = {v0, 0, t0, v1, 0, t1};
#pragma unroll
    for (int k = 0; k < 6; ++k) {
        unsigned long long x = c[k];
        for (int off = 32; off > 0; off >>= 1) x += __shfl_xor(x, off, 64);
        if (lane_id() == 0) atomicAdd(&stats[k], x);
    }
}

__global__ void k_zero_u64(unsigned long long* p, int count) {
    for (int i = threadIdx.x; i < count; i += blockDim.x) p[i] = 0;
}

__global__ void k_zero_counter(int32_t* counter) { *counter = 0; }

__global__ __launch_bounds__(kCopyBlock) void k_copy16(const int4* __restrict__ src, int4* __restrict__ dst,
                                                       size_t count) {
    for (size_t i = size_t(blockIdx.x) * kCopyBlock + threadIdx.x; i < count; i += size_t(gridDim.x) * kCopyBlock)
        dst[i] = src[i];
}

// Overlap, level by level. A workgroup takes kOvQueries query boxes (in the
// query tree's Morton order) and keeps in LDS the (query, sibling pair) items
// of one tree level: each step tests both children of every item with one
// 64-byte pair load (two items per lane in flight), collects the overlapping
// leaves and lists the entered internal children for the next level. A query's
// dependent chain is thus the tree depth, and the loads of a level are
// independent. An item whose child finds the next list full walks that child's
// subtree at once in preorder. Pairs collect in LDS and go out with one atomic
// per workgroup at the end (directly, one wave-wide atomic per step, once the
// LDS buffer is full). Every leaf whose box overlaps the query box is reached
// (an ancestor's box contains its descendants'), so the pair set is that of
// the per-query walk of src/bvh/bvh_overlap.cu:25-251, and the counter keeps
// counting past max_pairs so the caller gets the exact total (:209-214).
// LDS per workgroup: the two item lists (kOvCap entries of 5 bytes each) and
// the pair buffer (8 bytes an entry) set how many workgroups share a CU. On the
// 1M-triangle self query: lists 2048 / buffer 2048 (40 KiB) 334 us, 2048 / 512
// 290 us, 1024 / 1024 236 us, 1024 / 512 (17 KiB) 222 us, and smaller sizes
// the same 221-222 us.
constexpr int kOvThreads = 256;
constexpr int kOvQueries = 128;
constexpr int kOvCap = 1024;
constexpr int kOvPairBuf = 512;

struct OvShared {
    lux_aabb qb[kOvQueries];
    int32_t qid[kOvQueries];
    uint32_t item[2][kOvCap];  // pair slot (children at slot, slot + 1)
    uint8_t iq[2][kOvCap];     // query within the workgroup
    lux_pair out[kOvPairBuf];
    uint32_t count[2];
    uint32_t nout;
    int32_t base;
};

__device__ __forceinline__ void emit_global(bool emit, int a, int b, lux_pair* __restrict__ pairs, int max_pairs,
                                            int32_t* counter) {
    const uint64_t m = ballot64(emit);
    if (!m) return;
    const uint32_t leader = uint32_t(__ffsll((unsigned long long)m) - 1);
    int base = 0;
    if (lane_id() == leader)
        base = __hip_atomic_fetch_add(counter, int(__popcll(m)), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    base = __shfl(base, int(leader), 64);
    if (emit) {
        const int idx = base + int(__popcll(m & lanemask_lt()));
        if (idx < max_pairs) {
            lux_pair pr;
            pr.a = a;
            pr.b = b;
            pairs[idx] = pr;
        }
    }
}

// One pair found by this lane (emit) goes to the workgroup's LDS buffer, or
// out directly once the buffer is full.
__device__ __forceinline__ void emit_pair(OvShared& sh, bool emit, int a, int b, lux_pair* __restrict__ pairs,
                                          int max_pairs, int32_t* counter) {
    bool spill = false;
    if (emit) {
        const uint32_t at = __hip_atomic_fetch_add(&sh.nout, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        if (at < uint32_t(kOvPairBuf)) {
            lux_pair pr;
            pr.a = a;
            pr.b = b;
            sh.out[at] = pr;
        } else {
            spill = true;
        }
    }
    if (ballot64(spill)) emit_global(spill, a, b, pairs, max_pairs, counter);
}

__device__ __forceinline__ bool node_overlap(const float4& a, const float4& b, const lux_aabb& q) {
    return box_overlap(a.x, a.y, a.z, a.w, b.x, b.y, q);
}

// Preorder walk of the subtree at `slot` (an internal node already known to
// overlap), ending at the node's escape.
__device__ void overlap_subtree(OvShared& sh, const lux_bvh_node* __restrict__ nodes, uint32_t nc, uint32_t slot,
                                uint32_t stop, const lux_aabb& qb, int qid, int self_mode,
                                lux_pair* __restrict__ pairs, int max_pairs, int32_t* counter, DevInfo* info) {
    uint32_t k = slot;
    for (uint32_t guard = 0; guard <= nc; ++guard) {
        float4 a, b;
        load_node32(nodes, k, a, b);
        const int prim = __float_as_int(b.z);
        const bool hit = node_overlap(a, b, qb);
        emit_pair(sh, hit && prim >= 0 && (!self_mode || prim > qid), self_mode ? qid : prim,
                  self_mode ? prim : qid, pairs, max_pairs, counter);
        k = (hit && prim < 0) ? uint32_t(~prim) : __float_as_uint(b.w);
        if (k == stop || k >= nc) return;
    }
    set_error(info, kErrWalkOrder);
}

// Both children of one item: leaves to the pair buffer, entered internal
// children to the next level's list.
__device__ __forceinline__ void overlap_item(OvShared& sh, int nxt, bool valid, uint32_t c, int qi,
                                             const float4& a0, const float4& b0, const float4& a1, const float4& b1,
                                             const lux_bvh_node* __restrict__ nodes, uint32_t nc, int self_mode,
                                             lux_pair* __restrict__ pairs, int max_pairs, int32_t* counter,
                                             DevInfo* info) {
    const lux_aabb qb = sh.qb[qi];
    const int qid = sh.qid[qi];
    const int p0 = __float_as_int(b0.z), p1 = __float_as_int(b1.z);
    const bool h0 = valid && node_overlap(a0, b0, qb), h1 = valid && node_overlap(a1, b1, qb);
    emit_pair(sh, h0 && p0 >= 0 && (!self_mode || p0 > qid), self_mode ? qid : p0, self_mode ? p0 : qid, pairs,
              max_pairs, counter);
    emit_pair(sh, h1 && p1 >= 0 && (!self_mode || p1 > qid), self_mode ? qid : p1, self_mode ? p1 : qid, pairs,
              max_pairs, counter);
#pragma unroll
    for (int j = 0; j < 2; ++j) {
        const int p = j ? p1 : p0;
        if (!(j ? h1 : h0) || p >= 0) continue;
        const uint32_t child = uint32_t(~p);
        if (child + 1 >= nc) {
            set_error(info, kErrWalkOrder);
            continue;
        }
        const uint32_t at = __hip_atomic_fetch_add(&sh.count[nxt], 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        if (at < uint32_t(kOvCap)) {
            sh.item[nxt][at] = child;
            sh.iq[nxt][at] = uint8_t(qi);
        } else {
            overlap_subtree(sh, nodes, nc, c + uint32_t(j), __float_as_uint(j ? b1.w : b0.w), qb, qid, self_mode,
                            pairs, max_pairs, counter, info);
        }
    }
}

__global__ __launch_bounds__(kOvThreads) void k_overlap(const lux_bvh_node* __restrict__ nodes, int node_count,
                                                        const lux_aabb* __restrict__ qboxes,
                                                        const int32_t* __restrict__ qids,
                                                        const uint32_t* __restrict__ qorder, int nq, int self_mode,
                                                        lux_pair* __restrict__ pairs, int max_pairs, int32_t* counter,
                                                        DevInfo* info) {
    __shared__ OvShared sh;
    const uint32_t nc = uint32_t(node_count);
    const int q0 = blockIdx.x * kOvQueries;
    const int nql = min(kOvQueries, nq - q0);
    const int tid = threadIdx.x;
    if (tid < 2) sh.count[tid] = 0;
    if (tid == 0) sh.nout = 0;
    __syncthreads();

    // the root: slot 0, alone
    {
        float4 a, b;
        load_node32(nodes, 0, a, b);
        const int prim = __float_as_int(b.z);
        bool emit = false;
        int qid = -1;
        if (tid < nql) {
            const uint32_t src = qorder[q0 + tid];
            const lux_aabb qb = qboxes[src];
            qid = qids[src];
            sh.qb[tid] = qb;
            sh.qid[tid] = qid;
            if (node_overlap(a, b, qb)) {
                if (prim >= 0) {
                    emit = !self_mode || prim > qid;
                } else if (uint32_t(~prim) + 1 < nc) {
                    const uint32_t at = __hip_atomic_fetch_add(&sh.count[0], 1u, __ATOMIC_RELAXED,
                                                               __HIP_MEMORY_SCOPE_WORKGROUP);
                    sh.item[0][at] = uint32_t(~prim);  // at < kOvQueries <= kOvCap
                    sh.iq[0][at] = uint8_t(tid);
                } else {
                    set_error(info, kErrWalkOrder);
                }
            }
        }
        emit_pair(sh, emit, self_mode ? qid : prim, self_mode ? prim : qid, pairs, max_pairs, counter);
    }
    __syncthreads();

    for (int cur = 0;; cur ^= 1) {
        const uint32_t count = min(sh.count[cur], uint32_t(kOvCap));
        if (count == 0) break;
        __syncthreads();  // every thread has read the count
        const int nxt = cur ^ 1;
        if (tid == 0) sh.count[nxt] = 0;
        __syncthreads();
        for (uint32_t it = uint32_t(tid); it < count; it += 2 * kOvThreads) {
            const uint32_t it2 = it + kOvThreads;
            const bool two = it2 < count;
            const uint32_t c0 = sh.item[cur][it], c1 = two ? sh.item[cur][it2] : c0;
            const int q0i = sh.iq[cur][it], q1i = two ? sh.iq[cur][it2] : q0i;
            float4 a00, b00, a01, b01, a10, b10, a11, b11;
            load_node32(nodes, c0, a00, b00);
            load_node32(nodes, c0 + 1, a01, b01);
            load_node32(nodes, c1, a10, b10);
            load_node32(nodes, c1 + 1, a11, b11);
            overlap_item(sh, nxt, true, c0, q0i, a00, b00, a01, b01, nodes, nc, self_mode, pairs, max_pairs, counter,
                         info);
            overlap_item(sh, nxt, two, c1, q1i, a10, b10, a11, b11, nodes, nc, self_mode, pairs, max_pairs, counter,
                         info);
        }
        __syncthreads();  // the next list is complete
    }

    // flush the buffered pairs: one atomic for the workgroup
    const uint32_t nout = min(sh.nout, uint32_t(kOvPairBuf));
    if (tid == 0)
        sh.base = nout ? __hip_atomic_fetch_add(counter, int(nout), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) : 0;
    __syncthreads();
    for (uint32_t i = uint32_t(tid); i < nout; i += kOvThreads) {
        const int64_t idx = int64_t(sh.base) + int64_t(i);
        if (idx < max_pairs) pairs[idx] = sh.out[i];
    }
}

}  // namespace

namespace {
// Below kOrderMinRays rays the origin sort costs more than the locality it buys.
const uint32_t* maybe_order(const BvhDev& d, RaySortDev* order, const lux_ray* rays, int n, hipStream_t s) {
    if (!order || n < kOrderMinRays || d.n < 2) return nullptr;
    return ray_order(*order, d, rays, n, s);
}

}  // namespace

const uint32_t* closest_order(RaySortDev& r, bool sort, const BvhDev& d, const lux_ray* rays, int n,
                              hipStream_t s) {
    return maybe_order(d, sort ? &r : nullptr, rays, n, s);
}

namespace {
RayTree ray_tree(const BvhDev& d) {
    RayTree t;
    t.nodes = d.nodes;
    t.wide = d.wide;
    t.wide_leaf = d.wide_leaf;
    t.node_count = d.n > 0 ? 2 * d.n - 1 : 0;
    t.records = (d.n > 1 && uint32_t(d.n) <= kMaxWideRecords) ? uint32_t(d.n - 1) : 0u;
    return t;
}
}  // namespace

namespace {
// Lanes per ray of a call of n rays (k_trace_parts): where the calls that leave
// the chip idle end. Closest hit, 1 / 4 / 8 / 16 lanes: 2^14 rays in 2^20 random
// triangles (with their build) 884 / 648 / 590 / 569 us, 2^15 395 / 165 / 123 /
// 135, 2^16 in 2^18 (with the refit) 431 / 260 / 257 / 283; 2^17 in 500 000
// 382 / 277 / 285, on a sphere mesh 133 / 119 / 122; at 2^18 one lane is the
// best for the soup (422 / 455) and within 6 % on the sphere.
int lanes_per_ray(const RayTree& tree, int n) {
    if (tree.records == 0) return 1;
    return n <= (1 << 14) ? 16 : n <= (1 << 16) ? 8 : n <= (1 << 17) ? 4 : 1;
}

template <bool kAny>
void launch_trace(const char* name, const BvhDev& d, const uint32_t* order, const lux_triangle* tris, int tri_count,
                  const lux_ray* rays, int n, void* out, hipStream_t s) {
    const RayTree tree = ray_tree(d);
    const int group = lanes_per_ray(tree, n);
    if (group > 1)
        LUX_LAUNCH(name, k_trace_parts<kAny>, div_up(int64_t(n) * group, kBlock), kBlock, 0, s, tree, tris, tri_count,
                   rays, n, order, group, out, d.info);
    else
        LUX_LAUNCH(name, k_trace<kAny>, div_up(n, kBlock), kBlock, 0, s, tree, tris, tri_count, rays, n, order, out,
                   d.info);
}
}  // namespace

void trace_closest(const BvhDev& d, const uint32_t* order, const lux_triangle* tris, int tri_count,
                   const lux_ray* rays, int n, lux_hit* hits, hipStream_t s) {
    if (n <= 0) return;
    launch_trace<false>("trace_closest", d, order, tris, tri_count, rays, n, hits, s);
}

void trace_any(const BvhDev& d, RaySortDev* order, const lux_triangle* tris, int tri_count, const lux_ray* rays,
               int n, uint8_t* occluded, hipStream_t s) {
    if (n <= 0) return;
    launch_trace<true>("trace_any", d, maybe_order(d, order, rays, n, s), tris, tri_count, rays, n, occluded, s);
}

void trace_stats(const BvhDev& d, const lux_triangle* tris, int tri_count, const lux_ray* rays, int n,
                 unsigned long long* d_stats, hipStream_t s) {
    LUX_LAUNCH("trace_stats_zero", k_zero_u64, 1, 64, 0, s, d_stats, 6);
    if (n <= 0 || d.n <= 0) return;
    LUX_LAUNCH("trace_stats", k_trace_stats, div_up(n, kBlock), kBlock, 0, s, ray_tree(d), tris, tri_count, rays, n,
               d_stats, d.info);
}

void copy_device(void* dst, const void* src, size_t bytes, hipStream_t s) {
    size_t count = bytes / 16;
    if (count == 0) return;
    int grid = int(std::min<size_t>((count + kCopyBlock - 1) / kCopyBlock, 4096));
    LUX_LAUNCH("copy16", k_copy16, grid, kCopyBlock, 0, s, static_cast<const int4*>(src), static_cast<int4*>(dst),
               count);
}

void overlap_query(const BvhDev& tree, const BvhDev& queries, bool self_mode, int max_pairs,
                   lux_pair* pairs, int32_t* counter, hipStream_t s) {
    LUX_LAUNCH("overlap_zero", k_zero_counter, 1, 1, 0, s, counter);
    if (tree.n <= 0 || queries.n <= 0 || max_pairs <= 0) return;
    const int slots = tree.n > 1 ? 2 * tree.n : 1;  // sibling-pair array
    LUX_LAUNCH(self_mode ? "overlap_self" : "overlap_cross", k_overlap, div_up(queries.n, kOvQueries), kOvThreads,
               0, s, (const lux_bvh_node*)tree.pairs, slots, (const lux_aabb*)queries.boxes,
               (const int32_t*)queries.ids, (const uint32_t*)queries.vals[0], queries.n, self_mode ? 1 : 0, pairs,
               max_pairs, counter, tree.info);
}

}  // namespace lux
