// two_level.hpp -- two-level (instanced) scenes: one LBVH per mesh over its
// object-space triangles (BLAS) and one over the instances' world bounds
// (TLAS), the layout of the reference's PreparedScene
// (src/scene/prepared_scene.cu:59-78, src/scene/scene_prepare.h:420-462).
#pragma once

#include <vector>

#include "lux_runtime.hpp"
#include "wide.hpp"

namespace lux {

// One mesh as the walks see it: its BLAS (right-first preorder nodes and the
// four-child records' leaf positions) and its triangles (object space, a slice of
// the scene's soup).
struct DevMesh {
    const lux_bvh_node* nodes;
    const lux_triangle* tris;
    const int32_t* wide_leaf;  // preorder position of each leaf child (4 * record + child)
    int32_t node_count;        // 2 n - 1 (0: empty mesh)
    int32_t tri_count;
};

// One instance: Transform::inv (row-major 4x4), the scene ordinal of its local
// triangle 0 (GpuSceneInstance::first_primitive, src/scene/gpu_scene.h:149-172),
// the preorder position of its TLAS leaf (-1: none) and, copied from its mesh so
// that entering the instance is one dependent load, the mesh's records and
// triangles.
struct DevInstance {
    float inv[16];
    const WideNode* wide;
    const lux_triangle* tris;
    int32_t tri_count;
    int32_t first;
    int32_t mesh;
    int32_t tlas_pos;
};
static_assert(sizeof(DevInstance) == 96, "instance record");

// What the walk kernels take by value.
struct TwoLevelView {
    const lux_bvh_node* tlas_nodes;  // the TLAS in right-first preorder, the reference's boxes
    const WideNode* tlas_wide;       // its records over tighter culling boxes (see TwoLevelDev)
    const DevInstance* instances;
    const DevMesh* meshes;
    DevInfo* info;
    int32_t tlas_node_count, instance_count, mesh_count;
    uint32_t tlas_records;
    uint32_t step_limit;  // TLAS nodes + the BLAS nodes of every instance: no walk takes more steps
};

// ---- device walk ------------------------------------------------------------------
// transform_point / transform_vector (src/core/mat4.cuh:173-203): row-major
// rows summed left to right; a point divides by w unless w == 1.
__device__ __forceinline__ f3 xform_point(const float* m, const f3& p) {
    const float x = m[0] * p.x + m[1] * p.y + m[2] * p.z + m[3];
    const float y = m[4] * p.x + m[5] * p.y + m[6] * p.z + m[7];
    const float z = m[8] * p.x + m[9] * p.y + m[10] * p.z + m[11];
    const float w = m[12] * p.x + m[13] * p.y + m[14] * p.z + m[15];
    return (w == 1.0f) ? make3(x, y, z) : make3(x / w, y / w, z / w);
}

__device__ __forceinline__ f3 xform_vector(const float* m, const f3& v) {
    return make3(m[0] * v.x + m[1] * v.y + m[2] * v.z, m[4] * v.x + m[5] * v.y + m[6] * v.z,
                 m[8] * v.x + m[9] * v.y + m[10] * v.z);
}

// A world ray in an instance's object space (inv: 16-byte aligned).
__device__ __forceinline__ void xform_ray(const float* inv, const f3& WO, const f3& WD, f3& O, f3& D) {
    float m[16];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const float4 row = reinterpret_cast<const float4*>(inv)[i];
        m[4 * i] = row.x;
        m[4 * i + 1] = row.y;
        m[4 * i + 2] = row.z;
        m[4 * i + 3] = row.w;
    }
    O = xform_point(m, WO);
    D = xform_vector(m, WD);
}

struct TwoLevelHit {
    int prim = -1, instance = -1, local = -1;
    float t = 0, u = 0, v = 0;
};

// The preorder walk is one flat loop over two levels. A lane starts in the TLAS (world
// ray); at an instance leaf it switches to that mesh's BLAS with the ray moved
// to object space and keeps the TLAS escape of the leaf; when the BLAS walk
// ends it returns to that escape with the world ray. One loop keeps the lanes
// of a wave in step whichever level each is on. t_max is shared by both
// levels: the reference gives the BLAS walk t_max = the current hit and keeps a
// BLAS hit only when it is nearer, which every hit the BLAS walk accepts is
// (it only accepts t < t_max), so updating t_max at once is the same.
// `any` stops at the first accepted triangle. `ignore` is a scene ordinal
// (should_skip_primitive) or -1.
template <typename World>
__device__ __forceinline__ TwoLevelHit two_level_walk(const TwoLevelView& s, World&& world, float t_min, float t_max,
                                                      bool any, int ignore) {
    f3 O, D;
    world(O, D);
    SlabRay sr = make_slab_ray(O, D, t_min);
    const lux_bvh_node* nodes = s.tlas_nodes;
    uint32_t nc = uint32_t(s.tlas_node_count);
    const lux_triangle* tris = nullptr;
    int tcount = 0, first = -1, inst_cur = -1, ignore_local = -1;
    bool in_blas = false;
    uint32_t resume = 0;
    uint32_t k = 0;
    uint32_t steps = s.step_limit;
    TwoLevelHit best;
    for (;;) {
        if (k >= nc) {
            if (!in_blas) break;
            in_blas = false;  // back to the TLAS at the instance leaf's escape
            nodes = s.tlas_nodes;
            nc = uint32_t(s.tlas_node_count);
            k = resume;
            world(O, D);
            sr = make_slab_ray(O, D, t_min);
            continue;
        }
        if (steps-- == 0u) {
            set_error(s.info, kErrWalkOrder);
            break;
        }
        float4 a, b;
        load_node(nodes, int(k), a, b);
        const int prim = __float_as_int(b.z);
        const uint32_t esc = __float_as_uint(b.w);
        // the branch-free test unless some active lane's current ray (world or
        // object space) has an axis-parallel component; a wave-uniform choice
        const bool any_parallel = wave_any_parallel(sr);
        const bool pass = any_parallel ? slab_hit(sr, t_max, a.x, a.y, a.z, a.w, b.x, b.y)
                                       : slab_hit_np(sr, t_max, a.x, a.y, a.z, a.w, b.x, b.y);
        if (!pass) {
            k = esc;
            continue;
        }
        if (prim < 0) {
            ++k;  // the right child
            continue;
        }
        k = esc;
        if (!in_blas) {  // instance leaf: enter its BLAS if it has one
            if (prim >= s.instance_count) continue;
            const DevInstance& in = s.instances[prim];
            if (in.tri_count <= 0 || in.first < 0) continue;
            resume = esc;
            in_blas = true;
            nodes = s.meshes[in.mesh].nodes;
            nc = uint32_t(s.meshes[in.mesh].node_count);
            tris = in.tris;
            tcount = in.tri_count;
            first = in.first;
            inst_cur = prim;
            ignore_local = (ignore >= first && ignore - first < tcount) ? ignore - first : -1;
            const f3 WO = O, WD = D;
            xform_ray(in.inv, WO, WD, O, D);
            sr = make_slab_ray(O, D, t_min);
            k = 0;
            continue;
        }
        if (prim == ignore_local) continue;  // should_skip_primitive
        if (prim >= tcount) {
            set_error(s.info, kErrPrimRange);
            continue;
        }
        const float* p = reinterpret_cast<const float*>(tris + prim);
        const f3 v0 = make3(p[0], p[1], p[2]), v1 = make3(p[3], p[4], p[5]), v2 = make3(p[6], p[7], p[8]);
        float t, u, v;
        if (tri_hit(O, D, t_min, t_max, v0, v1, v2, t, u, v)) {
            t_max = t;
            best.prim = first + prim;
            best.instance = inst_cur;
            best.local = prim;
            best.t = t;
            best.u = u;
            best.v = v;
            if (any) break;
        }
    }
    return best;
}

// The same queries by the four-child records of both levels (wide.hpp), near child
// first on one LDS stack. A TLAS step enters records and instance leaves alike, in
// the order of their entries; taking an instance leaf moves the ray to object
// space and walks that BLAS above the entry depth of the stack, returning to the
// world ray when the stack falls back to it. The triangle tests and the instance
// entries (a matrix transform and three correctly rounded quotients) are gathered
// across the wave: a lane that holds passed leaf children or an instance waits
// until a quarter of the working lanes hold some.
// The preorder walk above visits triangles in the order (TLAS preorder of the
// instance leaf, BLAS preorder of the triangle leaf) and keeps the first of equal
// t; this walk keeps, of equal t, the one smallest in that order. The TLAS records
// hold the culling boxes (see TwoLevelDev), every byte box only culls, and at the
// end the winner's own boxes -- its BLAS leaf in object space and its instance's
// TLAS leaf, the reference's box, in world space -- are tested the reference's way
// with both entries at most t: the check of wide.hpp over both levels. An any-hit
// query ends at its first hit and asks only that both boxes are entered before
// t_max. world(o, d) gives the ray. Returns false when the preorder walk has to
// decide (the check fails, the stack is full, the arrays are malformed).
// A ray on `group` lanes: parts of it as in wide_query; an instance's culling box
// holds its geometry at every t, so a triangle's boxes of both levels are met in
// the same part.
// 2^22 rays over 64 instances of 2^16 triangles: closest 8.1 ms, occlusion 6.7 ms;
// by sibling pairs 18.8 (near child first, one lane's entries at a time) and 11.9 ms
// (preorder, gathered). 1000 rays over 40 instances of 5000: 105 us against 422.
// kReload: the view is in memory and read again at each use, so that its fields
// take no registers through the walk.
template <bool kReload, typename World>
__device__ __forceinline__ bool two_level_wide(const TwoLevelView& view, World&& world, float t_min, float t_bound,
                                               bool any, int ignore, int group, int part, uint32_t* stack,
                                               int stride, TwoLevelHit& best) {
    constexpr uint32_t kNone = 0x7fffffffu;
    best = TwoLevelHit{};
    auto fields = [&]() -> const TwoLevelView& {
        const TwoLevelView* p = &view;
        if (kReload) asm volatile("" : "+v"(p));
        return *p;
    };
    const TwoLevelView& s = view;
    if (s.tlas_node_count == 0) return true;
    f3 O = make3(0, 0, 0), D = O;
    SlabRay sr = {};
    bool stale = true;  // sr is not the ray of the next step
    float lo = t_min, hi = t_bound;
    bool skip = false;
    if (group > 1) {
        world(O, D);
        skip = !ray_part(s.tlas_nodes, make_slab_ray(O, D, t_min), group, part, lo, hi);
    }
    float t_max = t_bound;
    float t_cull = wide_bound(hi);
    const WideNode* wide = s.tlas_wide;
    uint32_t records = s.tlas_records;
    // the next record, kLeafBit | instance, or kNone: the top of the stack
    uint32_t item = records ? 0u : kLeafBit | uint32_t(s.tlas_nodes[0].primitive_id);
    uint32_t hc = 0, hmask = 0;
    uint4 ref = make_uint4(0, 0, 0, 0);
    int sp = 0, sp0 = 0;
    const lux_triangle* tris = nullptr;
    int inst = -1, ignore_local = -1;
    int best_inst = -1, best_local = -1;
    uint32_t best_at = 0;
    uint32_t steps = s.step_limit;
    bool in_blas = false, done = skip, failed = false;
    auto leaf = [&](uint32_t at, uint32_t r) {
        const uint32_t prim = r & kIndexMask;
        if (int(prim) == ignore_local || r == kWideEmpty) return false;  // should_skip_primitive
        if (prim > records) {  // a BLAS of `records` records has one triangle more
            set_error(fields().info, kErrPrimRange);
            return false;
        }
        const float* p = reinterpret_cast<const float*>(tris + prim);
        float t, u, v;
        if (!tri_uvt(O, D, make3(p[0], p[1], p[2]), make3(p[3], p[4], p[5]), make3(p[6], p[7], p[8]), t, u, v) ||
            !(t > t_min))
            return false;
        bool take = t < t_max;
        if (!take && !any && best_inst >= 0 && t == t_max) {  // exact tie: the smaller (TLAS, BLAS) preorder position
            if (inst != best_inst) {
                take = fields().instances[inst].tlas_pos < fields().instances[best_inst].tlas_pos;
            } else if (records) {
                const int32_t* pos = fields().meshes[fields().instances[inst].mesh].wide_leaf;
                take = pos[at] < pos[best_at];
            }
        }
        if (!take) return false;
        best_inst = inst;
        best_local = int(prim);
        best_at = at;
        if (any) return true;
        t_max = t;
        t_cull = fminf(t_cull, t + fabsf(t) * kSoftWindow);
        return false;
    };
    for (;;) {
        if (!done & (hmask == 0) & !(item & kLeafBit)) {
            if (item == kNone) {
                if (in_blas && sp == sp0) {  // leave the instance
                    in_blas = false;
                    stale = true;
                }
                if (sp == 0)
                    done = true;
                else
                    item = stack[--sp * stride];
            }
            if (!done & !stale & !(item & kLeafBit)) {
                if (item >= records || steps-- == 0u) {
                    set_error(fields().info, kErrWalkOrder);
                    failed = done = true;
                } else {
                    float4 a, b, q;
                    load_wide(wide, item, a, b, q, ref);
                    float key[4];
                    bool pass[4];
                    wide_boxes<true>(a, b, q, sr, t_cull, key, pass);
                    uint32_t kid[4] = {ref.x, ref.y, ref.z, ref.w};
                    uint32_t mask = 0;
#pragma unroll
                    for (int k = 0; k < 4; ++k) {
                        const bool tri = in_blas & (int32_t(kid[k]) < 0);
                        const bool empty = kid[k] == kWideEmpty;
                        key[k] = (pass[k] & !tri & !empty) ? key[k] : INFINITY;
                        mask |= (pass[k] & tri) ? (1u << k) : 0u;
                    }
                    hc = item;
                    hmask = mask;
                    item = kNone;
                    wide_sort(key, kid);
                    if (key[0] < INFINITY) {
                        item = kid[0];
                        const bool p1 = key[1] < INFINITY, p2 = key[2] < INFINITY, p3 = key[3] < INFINITY;
                        if (sp + int(p1) + int(p2) + int(p3) > kWideStack) {
                            failed = done = true;
                            hmask = 0;
                        } else {
                            if (p3) stack[sp++ * stride] = kid[3];
                            if (p2) stack[sp++ * stride] = kid[2];
                            if (p1) stack[sp++ * stride] = kid[1];
                        }
                    }
                }
            }
        }
        const bool holds = !done & (stale | (hmask != 0) | ((item & kLeafBit) != 0));
        const uint64_t want = __ballot(holds);
        const uint64_t more = __ballot(!done & !holds);
        if (!more) {
            if (!want) break;
        } else if (__popcll(want) * kGatherDiv < __popcll(want | more)) {
            continue;
        }
        while (hmask) {
            const uint32_t k = uint32_t(__ffs(int(hmask))) - 1u;
            hmask &= hmask - 1u;
            const uint32_t r0 = (k & 1u) ? ref.y : ref.x, r1 = (k & 1u) ? ref.w : ref.z;
            if (leaf(4u * hc + k, (k & 2u) ? r1 : r0)) {
                done = true;
                hmask = 0;
            }
        }
        if (group > 1) {  // the lanes of a ray tell each other
            float t = best_inst < 0 ? INFINITY : any ? -INFINITY : t_max;
            for (int off = 1; off < group; off <<= 1) t = fminf(t, __shfl_xor(t, off, 64));
            if (any)
                done |= t < INFINITY;
            else
                t_cull = fminf(t_cull, t + fabsf(t) * kSoftWindow);
        }
        if (!done && (stale | ((item & kLeafBit) != 0))) {  // only ever in the TLAS
            const TwoLevelView& s = fields();
            world(O, D);
            wide = s.tlas_wide;
            records = s.tlas_records;
            stale = false;
            const int next = item & kLeafBit ? int(item & kIndexMask) : -1;
            if (next >= 0) {
                item = kNone;
                stale = true;
            }
            if (uint32_t(next) < uint32_t(s.instance_count)) {
                const DevInstance& in = s.instances[next];
                const int tri_count = in.tri_count, first = in.first;
                if (tri_count > 0 && first >= 0) {
                    const f3 WO = O, WD = D;
                    xform_ray(in.inv, WO, WD, O, D);
                    inst = next;
                    in_blas = true;
                    stale = false;
                    sp0 = sp;
                    wide = in.wide;
                    records = uint32_t(tri_count) - 1u;
                    tris = in.tris;
                    ignore_local = (ignore >= first && ignore - first < tri_count) ? ignore - first : -1;
                    if (records) {
                        item = 0;
                    } else {  // one triangle
                        ref.x = kLeafBit;
                        hc = 0;
                        hmask = 1;
                    }
                }
            }
            sr = make_slab_ray(O, D, lo);
            if (!wide_takes(D) || records >= kMaxWideRecords) {
                failed = done = true;
                hmask = 0;
            }
        }
    }
    int at_inst = -1, at_tri = 0;  // the winner's leaves
    if (best_inst >= 0) {
        const TwoLevelView& s = fields();
        const DevInstance& in = s.instances[best_inst];
        at_inst = in.tlas_pos;
        at_tri = in.tri_count > 1 ? s.meshes[in.mesh].wide_leaf[best_at] : 0;
    }
    if (group > 1) {
        int fail = failed;
        for (int off = 1; off < group; off <<= 1) {
            fail |= __shfl_xor(fail, off, 64);
            const float t = __shfl_xor(t_max, off, 64);
            const int i = __shfl_xor(best_inst, off, 64), l = __shfl_xor(best_local, off, 64);
            const int ai = __shfl_xor(at_inst, off, 64), at = __shfl_xor(at_tri, off, 64);
            const bool first = ai < at_inst || (ai == at_inst && at < at_tri);
            if (i >= 0 && (best_inst < 0 || t < t_max || (t == t_max && first))) {
                t_max = t;
                best_inst = i;
                best_local = l;
                at_inst = ai;
                at_tri = at;
            }
        }
        failed = fail != 0;
    }
    if (failed) return false;
    if (best_inst < 0) return true;
    // the winner's boxes, and its u and v: the same operations on the same
    // operands as the leaf test that took it
    const TwoLevelView& v = fields();
    const DevInstance& in = v.instances[best_inst];
    const DevMesh& mesh = v.meshes[in.mesh];
    world(O, D);
    const float t_box = any ? t_bound : t_max;
    if (!wide_settled(v.tlas_nodes, v.tlas_node_count, at_inst, make_slab_ray(O, D, t_min), t_box, v.info)) return false;
    f3 o, d;
    xform_ray(in.inv, O, D, o, d);
    if (!wide_settled(mesh.nodes, mesh.node_count, at_tri, make_slab_ray(o, d, t_min), t_box, v.info)) return false;
    const float* p = reinterpret_cast<const float*>(in.tris + best_local);
    (void)tri_uvt(o, d, make3(p[0], p[1], p[2]), make3(p[3], p[4], p[5]), make3(p[6], p[7], p[8]), best.t, best.u,
                  best.v);
    best.prim = in.first + best_local;
    best.instance = best_inst;
    best.local = best_local;
    return true;
}

// ---- host side ----------------------------------------------------------------------
struct TwoLevelDev {
    std::vector<BvhDev> blas;  // per mesh (n = 0 for an empty mesh)
    // Over the non-empty instance world bounds, ids = instance ids. Its records are
    // made from culling nodes: each leaf box narrowed to its instance's world
    // bounds intersected with the world box of the mesh's bounding sphere
    // (center M c, half-extent r |row i of M| on axis i: the exact box of the
    // transformed sphere), both widened by what the instance's M inv may
    // deviate from the identity; internal boxes the unions of their children.
    BvhDev tlas;
    lux_bvh_node* tlas_cull = nullptr;
    int tlas_cull_capacity = 0, instance_capacity = 0;
    std::vector<float> mesh_sphere;  // per mesh: center xyz, radius (padded)
    lux_triangle* soup = nullptr;
    DevMesh* meshes = nullptr;
    DevInstance* instances = nullptr;
    std::vector<int32_t> mesh_tri_off;  // mesh_count + 1
    std::vector<lux_instance> host_instances;
    int mesh_count = 0, instance_count = 0, tlas_instances = 0;
    int64_t scene_primitives = 0;
    uint32_t step_limit = 0;
    size_t device_bytes = 0;
    bool whole = false;  // the instances, the TLAS and its records belong together
};

// Scene validation of one instance transform pair (src/scene/scene_validate.h:140-147,
// src/core/mat4.cuh:86-124): both matrices affine with |det3| > 1e-12 and
// m * inv, inv * m within 1e-4 of the identity.
bool instance_transform_valid(const float* m16, const float* inv16);
// make_transform's inverse and transform_bounds (src/core/mat4.cuh:126-159, 254-270).
void inverse_affine(const float* m16, float* inv16);
lux_aabb transform_bounds(const float* m16, const lux_aabb& b);

// Builds every BLAS and the TLAS (synchronous: validates, uploads, builds, waits).
void two_level_build(TwoLevelDev& s, const lux_triangle* tris, const int32_t* mesh_offsets, int mesh_count,
                     const lux_instance* instances, int instance_count, hipStream_t stream);
// New instance transforms / world bounds for the same meshes and instance count:
// rebuilds the TLAS and the instance records only. If that fails half way, views of the
// scene are refused until it succeeds.
void two_level_set_instances(TwoLevelDev& s, const lux_instance* instances, int instance_count,
                             hipStream_t stream);
void two_level_release(TwoLevelDev& s);
TwoLevelView two_level_view(const TwoLevelDev& s);

// Closest hit (or occlusion) of n device rays; ignore (nullable) holds one scene
// ordinal per ray that is skipped (-1: none). order (nullable): the rays in
// ray order, from two_level_order; results land at each ray's own index.
const uint32_t* two_level_order(RaySortDev& r, const TwoLevelDev& s, const lux_ray* rays, int n, hipStream_t stream);
void two_level_closest(const TwoLevelView& v, const uint32_t* order, const lux_ray* rays, const int32_t* ignore,
                       int n, lux_scene_hit* hits, hipStream_t stream);
void two_level_occluded(const TwoLevelView& v, const uint32_t* order, const lux_ray* rays, const int32_t* ignore,
                        int n, uint8_t* occluded, hipStream_t stream);

}  // namespace lux
