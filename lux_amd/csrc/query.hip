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

// One ray (wide.hpp): the records' walk, or the preorder walk where it hands the
// ray back.
template <bool kAny>
__device__ __forceinline__ WideHit trace_one(const RayTree& tree, const lux_triangle* __restrict__ tris,
                                             int tri_count, const RayIn& ray, int group, int part, uint32_t* stack,
                                             DevInfo* info, uint32_t& visits, uint32_t& tests) {
    // canonical from the start, so the loop's min/max need no per-step canonicalise
    const float t_max = __builtin_canonicalizef(ray.t_max);
    WideHit h = wide_query(tree, tris, tri_count, ray.o, ray.d, ray.t_min, t_max, kAny, -1, group, part, stack,
                           kBlock, info, visits, tests);
    if (h.failed && part == 0)
        h = preorder_query(tree, tris, tri_count, ray.o, ray.d, ray.t_min, t_max, kAny, -1, info, visits, tests);
    return h;
}

template <bool kAny>
__device__ __forceinline__ void store_result(void* __restrict__ out, int ray, const WideHit& found) {
    if (kAny) {
        static_cast<uint8_t*>(out)[ray] = found.prim >= 0 ? 1 : 0;
    } else {
        lux_hit h;
        h.primitive_id = found.prim;
        h.t = found.prim >= 0 ? found.t : INFINITY;
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
    uint32_t visits = 0, tests = 0;
    store_result<kAny>(out, ray, trace_one<kAny>(tree, tris, tri_count, load_ray(rays, ray), 1, 0, stack + threadIdx.x, info, visits, tests));
}

// Trees without records (one leaf, beyond 2^26 leaves): the preorder walk alone. One
// triangle, here / in k_trace: 1000 rays 3.6 / 3.8 us, 2^22 closest 27.8 / 28.4, any
// hit 24.9 / 25.4 (blocks of one wave 29.0 and 25.8).
constexpr int kPreorderBlock = 256;
template <bool kAny>
__global__ __launch_bounds__(kPreorderBlock) void k_trace_preorder(RayTree tree, const lux_triangle* __restrict__ tris,
                                                           int tri_count, const lux_ray* __restrict__ rays, int n,
                                                           const uint32_t* __restrict__ order, void* __restrict__ out,
                                                           DevInfo* info) {
    const int i = int(xcd_block()) * kPreorderBlock + threadIdx.x;
    if (i >= n) return;
    const int ray = order ? int(order[i]) : i;
    if (uint32_t(ray) >= uint32_t(n)) {
        set_error(info, kErrSpinLimit);
        return;
    }
    uint32_t visits = 0, tests = 0;
    const RayIn r = load_ray(rays, ray);
    store_result<kAny>(out, ray, preorder_query(tree, tris, tri_count, r.o, r.d, r.t_min,
                                                __builtin_canonicalizef(r.t_max), kAny, -1, info, visits, tests));
}

// Few rays: `group` lanes (a power of two) walk one ray (wide_query).
template <bool kAny>
__global__ __launch_bounds__(kBlock) __attribute__((amdgpu_waves_per_eu(kAny ? 7 : 6))) void k_trace_parts(
    RayTree tree, const lux_triangle* __restrict__ tris, int tri_count, const lux_ray* __restrict__ rays, int n,
    const uint32_t* __restrict__ order, int group, void* __restrict__ out, DevInfo* info) {
    __shared__ uint32_t stack[kWideStack * kBlock];
    const int i = (int(xcd_block()) * kBlock + int(threadIdx.x)) / group;
    if (i >= n) return;  // whole groups
    const int part = int(threadIdx.x) & (group - 1);
    const int ray = order ? int(order[i]) : i;
    if (uint32_t(ray) >= uint32_t(n)) {
        set_error(info, kErrSpinLimit);
        return;
    }
    uint32_t visits = 0, tests = 0;
    const WideHit h = trace_one<kAny>(tree, tris, tri_count, load_ray(rays, ray), group, part, stack + threadIdx.x, info, visits, tests);
    if (part == 0) store_result<kAny>(out, ray, h);
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
        const RayIn r = load_ray(rays, i);
        (void)trace_one<false>(tree, tris, tri_count, r, 1, 0, stack + threadIdx.x, info, v0, t0);
        (void)trace_one<true>(tree, tris, tri_count, r, 1, 0, stack + threadIdx.x, info, v1, t1);
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
            uint32_t src = qorder[q0 + tid];
            if (src >= uint32_t(nq)) {  // only after a failed sort
                set_error(info, kErrSpinLimit);
                src = 0;
            }
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
template <bool kAny>
void launch_trace(const char* name, BvhDev& d, const uint32_t* order, const lux_triangle* tris, int tri_count,
                  const lux_ray* rays, int n, void* out, hipStream_t s) {
    tree_copies(d, kCopyRecords, s);
    const RayTree tree = ray_tree(d);
    const int group = tree.records >= kPartsMinRecords ? lanes_per_ray(uint32_t(n)) : 1;
    if (tree.records == 0)
        LUX_LAUNCH(name, k_trace_preorder<kAny>, div_up(n, kPreorderBlock), kPreorderBlock, 0, s, tree, tris, tri_count, rays, n, order,
                   out, d.info);
    else if (group > 1)
        LUX_LAUNCH(name, k_trace_parts<kAny>, div_up(int64_t(n) * group, kBlock), kBlock, 0, s, tree, tris, tri_count,
                   rays, n, order, group, out, d.info);
    else
        LUX_LAUNCH(name, k_trace<kAny>, div_up(n, kBlock), kBlock, 0, s, tree, tris, tri_count, rays, n, order, out,
                   d.info);
}
}  // namespace

void trace_closest(BvhDev& d, const uint32_t* order, const lux_triangle* tris, int tri_count,
                   const lux_ray* rays, int n, lux_hit* hits, hipStream_t s) {
    if (n <= 0) return;
    launch_trace<false>("trace_closest", d, order, tris, tri_count, rays, n, hits, s);
}

void trace_any(BvhDev& d, RaySortDev* order, const lux_triangle* tris, int tri_count, const lux_ray* rays,
               int n, uint8_t* occluded, hipStream_t s) {
    if (n <= 0) return;
    launch_trace<true>("trace_any", d, maybe_order(d, order, rays, n, s), tris, tri_count, rays, n, occluded, s);
}

void trace_stats(BvhDev& d, const lux_triangle* tris, int tri_count, const lux_ray* rays, int n,
                 unsigned long long* d_stats, hipStream_t s) {
    LUX_LAUNCH("trace_stats_zero", k_zero_u64, 1, 64, 0, s, d_stats, 6);
    if (n <= 0 || d.n <= 0) return;
    tree_copies(d, kCopyRecords, s);
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

void overlap_query(BvhDev& tree, const BvhDev& queries, bool self_mode, int max_pairs,
                   lux_pair* pairs, int32_t* counter, hipStream_t s) {
    LUX_LAUNCH("overlap_zero", k_zero_counter, 1, 1, 0, s, counter);
    if (tree.n <= 0 || queries.n <= 0 || max_pairs <= 0) return;
    tree_copies(tree, kCopyPairs, s);
    const int slots = tree.n > 1 ? 2 * tree.n : 1;  // sibling-pair array
    LUX_LAUNCH(self_mode ? "overlap_self" : "overlap_cross", k_overlap, div_up(queries.n, kOvQueries), kOvThreads,
               0, s, (const lux_bvh_node*)tree.pairs, slots, (const lux_aabb*)queries.boxes,
               (const int32_t*)queries.ids, (const uint32_t*)queries.vals[0], queries.n, self_mode ? 1 : 0, pairs,
               max_pairs, counter, tree.info);
}

}  // namespace lux
