// wide.hpp -- four-child traversal records of an LBVH and the near-child-first
// walk over them, with the hit the right-first preorder walk would return.
//
// Record i belongs to internal node i of the radix tree (Karras order; record 0
// is the root) and holds up to four descendants whose leaf ranges make up that
// node's: its two children, with the larger internal one (by box area) opened
// until there are four. Every internal node has its record, so each is made
// from the node array alone and a walk uses about half of them. A child's box
// is kept as six bytes in the record's own frame (org + scale * byte, faces
// moved outwards), so a record is 64 bytes: half the loads of two sibling pairs
// with 32-byte boxes, and half the dependent steps. In a CPU model (2^20 random
// triangles, random rays) near-first walks take 50 records (193 boxes) per ray
// against 100 pairs (200 boxes); the byte boxes account for 2 % of them.
//
// Box tests are conservative: a ray that passes a leaf's own box by the
// reference's slab test (src/core/aabb.cuh:84-109) passes every byte box above
// it. Per axis the walk forms near = byte * (scale * inv) + (org - o) * inv.
// With all roundings this is off the true distance by at most 2^-22 of
// |(org - o) * inv| plus 2^-14 of |scale * inv|; the second part is covered by
// moving each face outwards by at least 2^-10 of the scale (make_wide), the first
// by kWideSlack in the far faces' base. An axis the reference treats as parallel
// (|d| < 1e-12, origin inside the slab or not) compares the origin with the
// byte faces (wide_parallel; chosen per wave). A record with a face beyond 1e18 or not
// finite has org = NaN, and every comparison with NaN passes. Rays with a
// direction component beyond 1e18 (or NaN) take the preorder walk.
//
// Equal result. The preorder walk (src/bvh/bvh_device.cuh:59-87) accepts a
// triangle iff its leaf box passes with entry at most the held t and t < held t,
// in preorder, so it returns the smallest (t, preorder position) over the
// triangles whose leaf boxes pass -- as long as no triangle's t lies below its
// own leaf box's entry (rounded, an entry can lie a few hundred ulps above the
// Moller-Trumbore t of a hit at a vertex or edge on the face the ray enters).
// This walk tests every triangle of every leaf whose byte boxes pass up to
// t_cull = t_max + |t_max| kSoftWindow, without its leaf box, and keeps the
// smallest (t, preorder position) of all. At the end wide_settled tests the
// winner's own leaf box the reference's way. If it passes with its entry at
// most t, the preorder walk returns the same hit: every triangle with a smaller
// or equal t and a smaller position would have been held here instead, so none
// exists among the reached, and the preorder walk reaches the winner holding a
// larger t. Otherwise (a box missed by rounding, an entry above t, a box with a
// NaN bound) the ray is walked again in preorder. The observed gap between a
// hit and its leaf box's entry is below 2^-14.7 relative, the window 2^-11.
//
// A lane whose stack is full stops and reports overflow; its caller then runs the
// preorder walk for that ray.
#pragma once

#include "lux_runtime.hpp"
#include "ordered.hpp"

namespace lux {

// Loaded as four float4: org.xyz scale.x | scale.yz lo.xy | lo.z hi.xyz | ref.
struct alignas(64) WideNode {
    float org[3];
    float scale[3];
    uint32_t lo[3];  // byte k: child k's lower face
    uint32_t hi[3];
    uint32_t ref[4];  // record of an internal child, kLeafBit | primitive id, kWideEmpty
};
static_assert(sizeof(WideNode) == 64, "wide record");

constexpr uint32_t kWideEmpty = 0xffffffffu;
// Records are loaded at base + 32-bit byte offset, so a walk takes trees of at
// most this many leaves (4 GiB of records).
constexpr uint32_t kMaxWideRecords = 1u << 26;
constexpr float kWideSlack = 0x1p-20f;

// Record from up to four children (boxes and refs; `count` of them). Faces are
// rounded outwards by at least 2^-8 of the scale and org lies at least 2^-10 of
// it below the lowest face.
__device__ __forceinline__ void make_wide(WideNode& w, const lux_aabb* box, const uint32_t* ref, int count) {
#pragma unroll
    for (int k = 0; k < 4; ++k) w.ref[k] = k < count ? ref[k] : kWideEmpty;
    bool finite = true;
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        float lo[4], hi[4], mn = INFINITY, mx = -INFINITY;
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            lo[k] = a == 0 ? box[k].p_min.x : (a == 1 ? box[k].p_min.y : box[k].p_min.z);
            hi[k] = a == 0 ? box[k].p_max.x : (a == 1 ? box[k].p_max.y : box[k].p_max.z);
            if (k < count) {
                finite = finite && fabsf(lo[k]) < 1e18f && fabsf(hi[k]) < 1e18f;
                mn = fminf(mn, fminf(lo[k], hi[k]));
                mx = fmaxf(mx, fmaxf(lo[k], hi[k]));
            }
        }
        // the float below mn; 1e-30 below a zero or tiny one
        const float below = fabsf(mn) > 1e-30f ? mn - fabsf(mn) * 0x1.8p-24f : mn - 1e-30f;
        const float big = fmaxf(fabsf(mn), fabsf(mx));
        const float s = fmaxf(fmaxf((mx - below) * (1.0f / 253.0f), big * 1e-9f), 1e-20f);
        const float org = fminf(below, mn - s * 0x1p-10f);
        uint32_t ql = 0, qh = 0;
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const float l = floorf((lo[k] - org) / s - 0x1p-8f), h = ceilf((hi[k] - org) / s + 0x1p-8f);
            const uint32_t bl = k < count ? uint32_t(fminf(fmaxf(l, 0.0f), 255.0f)) : 255u;
            const uint32_t bh = k < count ? uint32_t(fminf(fmaxf(h, 0.0f), 255.0f)) : 0u;
            ql |= bl << (8 * k);
            qh |= bh << (8 * k);
        }
        w.org[a] = org;
        w.scale[a] = s;
        w.lo[a] = ql;
        w.hi[a] = qh;
    }
    if (!finite) w.org[0] = w.org[1] = w.org[2] = NAN;
}

__device__ __forceinline__ void store_wide(WideNode* dst, const WideNode& w) {
    float4* p = reinterpret_cast<float4*>(dst);
    p[0] = make_float4(w.org[0], w.org[1], w.org[2], w.scale[0]);
    p[1] = make_float4(w.scale[1], w.scale[2], __uint_as_float(w.lo[0]), __uint_as_float(w.lo[1]));
    p[2] = make_float4(__uint_as_float(w.lo[2]), __uint_as_float(w.hi[0]), __uint_as_float(w.hi[1]),
                       __uint_as_float(w.hi[2]));
    p[3] = make_float4(__uint_as_float(w.ref[0]), __uint_as_float(w.ref[1]), __uint_as_float(w.ref[2]),
                       __uint_as_float(w.ref[3]));
}

__device__ __forceinline__ WideNode empty_wide() {
    WideNode w;
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        w.org[a] = 0.0f;
        w.scale[a] = 1.0f;
        w.lo[a] = 0xffffffffu;  // an empty interval
        w.hi[a] = 0;
    }
#pragma unroll
    for (int k = 0; k < 4; ++k) w.ref[k] = kWideEmpty;
    return w;
}

// One thread per internal node: its two children, the larger internal one
// opened, then the largest of the three. Its reads are gathers of positions and
// 32-byte nodes close to each other (Karras order and preorder both follow the
// leaves), its write one 64-byte record and 16 bytes of leaf positions. A node
// whose links or positions are out of range (a damaged tree) gets a record without
// children, never what the memory held.
__device__ __forceinline__ void fill_wide(int n, int i, const uint32_t* __restrict__ left,
                                          const uint32_t* __restrict__ right,
                                          const int32_t* __restrict__ pre_internal,
                                          const int32_t* __restrict__ pre_leaf,
                                          const lux_bvh_node* __restrict__ nodes, WideNode* __restrict__ wide,
                                          int32_t* __restrict__ wide_leaf, DevInfo* info) {
    const int total = 2 * n - 1;
    lux_aabb box[4];
    uint32_t ref[4];
    int32_t pos[4];
    float area[4] = {-1.0f, -1.0f, -1.0f, -1.0f};
    bool bad = false;
    auto load = [&](int k, uint32_t c) {
        const uint32_t idx = c & kIndexMask;
        const bool leaf = c & kLeafBit;
        bad |= idx >= uint32_t(leaf ? n : n - 1);
        const int p = bad ? 0 : (leaf ? pre_leaf[idx] : pre_internal[idx]);
        bad |= uint32_t(p) >= uint32_t(total);
        float4 a, b;
        load_node(nodes, bad ? 0 : p, a, b);
        box[k].p_min = lux_vec3{a.x, a.y, a.z};
        box[k].p_max = lux_vec3{a.w, b.x, b.y};
        pos[k] = p;
        ref[k] = leaf ? (kLeafBit | uint32_t(__float_as_int(b.z))) : idx;
        const float dx = a.w - a.x, dy = b.x - a.y, dz = b.y - a.z;
        area[k] = leaf ? -1.0f : dx * dy + dy * dz + dz * dx;
    };
    load(0, left[i]);
    load(1, right[i]);
    int count = 2;
#pragma unroll
    for (int open = 0; open < 2; ++open) {
        int best = -1;
        float ba = -1.0f;
#pragma unroll
        for (int k = 0; k < 2 + open; ++k)
            if (area[k] > ba) {
                ba = area[k];
                best = k;
            }
        if (best < 0 || bad) continue;
        uint32_t c = 0;
#pragma unroll
        for (int k = 0; k < 2 + open; ++k)
            if (k == best) c = ref[k];
        const uint32_t cl = left[c], cr = right[c];
#pragma unroll
        for (int k = 0; k < 2 + open; ++k)
            if (k == best) load(k, cl);
        load(2 + open, cr);
        ++count;
    }
    if (bad) {
        set_error(info, kErrWalkOrder);
        store_wide(wide + i, empty_wide());
        reinterpret_cast<int4*>(wide_leaf)[i] = make_int4(-1, -1, -1, -1);
        return;
    }
#pragma unroll
    for (int k = 2; k < 4; ++k)
        if (k >= count) {
            box[k] = box[0];
            ref[k] = kWideEmpty;
            pos[k] = -1;
        }
    WideNode w;
    make_wide(w, box, ref, count);
    store_wide(wide + i, w);
    reinterpret_cast<int4*>(wide_leaf)[i] = make_int4(pos[0], pos[1], pos[2], pos[3]);
}

__device__ __forceinline__ void load_wide(const WideNode* nodes, uint32_t i, float4& a, float4& b, float4& c,
                                          uint4& r) {
    const char* p = reinterpret_cast<const char*>(nodes) + (i << 6);
    const float4* q = reinterpret_cast<const float4*>(p);
    a = q[0];
    b = q[1];
    c = q[2];
    r = reinterpret_cast<const uint4*>(p)[3];
}

__device__ __forceinline__ float byte_of(uint32_t w, int k) { return float((w >> (8 * k)) & 0xffu); }

// True when the walk below takes the ray (see above).
__device__ __forceinline__ bool wide_takes(const f3& d) {
    return (fabsf(d.x) < 1e18f) & (fabsf(d.y) < 1e18f) & (fabsf(d.z) < 1e18f);
}

// Where the walk's box entries end for a ray bound t (a ray's t_max).
__device__ __forceinline__ float wide_bound(float t) { return t + fabsf(t) * kWideSlack; }

// The winner (leaf node at preorder position pos, distance t): true when the
// preorder walk returns it too (see above). An any-hit query passes the ray's
// t_max as t: there the leaf box only has to be entered before it. A position out
// of range (a damaged tree) is an error, and the preorder walk decides.
__device__ __forceinline__ bool wide_settled(const lux_bvh_node* __restrict__ nodes, int node_count, int pos,
                                             const SlabRay& sr, float t, DevInfo* info) {
    if (uint32_t(pos) >= uint32_t(node_count)) {
        set_error(info, kErrWalkOrder);
        return false;
    }
    float4 a, b;
    load_node(nodes, pos, a, b);
    float tn;
    const bool pass = slab_near<true>(sr, INFINITY, a.x, a.y, a.z, a.w, b.x, b.y, tn);
    const bool nan = !(a.x <= INFINITY) | !(a.y <= INFINITY) | !(a.z <= INFINITY) | !(a.w <= INFINITY) |
                     !(b.x <= INFINITY) | !(b.y <= INFINITY);
    return pass && !(tn > t) && !nan;
}

// One axis of a record for a ray parallel to it: everywhere inside a child's slab,
// or nowhere. The origin's place in byte units, cut at 1024 either way, stands for
// the distances, times 2^116: inside, a face is at least 2^-10 away (see above),
// so the entry is below -2^105 and the exit beyond 2^105, more than any hit's
// distance (coordinates below 1e18, other components above 1e-12); outside by
// more than 2^-9, one of them is the other way round.
__device__ __forceinline__ void wide_parallel(bool par, float org, float scale, float o, float& s, float& base) {
    float r = (org - o) * __builtin_amdgcn_rcpf(scale);
    r = r > 1024.0f ? 1024.0f : r;
    r = r < -1024.0f ? -1024.0f : r;
    s = par ? 0x1p116f : s;
    base = par ? r * 0x1p116f : base;
}

// The four byte boxes of a record (its first three float4) against the ray: entry
// distances and whether they are met between the ray's t_min and t_cull. kPar:
// some axis may be parallel; its inv is 0 (no other is, see wide_takes) and signs
// are read from inv, so that the ray's six flags need no registers.
template <bool kPar>
__device__ __forceinline__ void wide_boxes(const float4& a, const float4& b, const float4& q, const SlabRay& r,
                                           float t_cull, float* key, bool* pass) {
    float sx = a.w * r.inv.x, sy = b.x * r.inv.y, sz = b.y * r.inv.z;
    float bx = (a.x - r.o.x) * r.inv.x, by = (a.y - r.o.y) * r.inv.y, bz = (a.z - r.o.z) * r.inv.z;
    if (kPar) {
        wide_parallel(r.inv.x == 0.0f, a.x, a.w, r.o.x, sx, bx);
        wide_parallel(r.inv.y == 0.0f, a.y, b.x, r.o.y, sy, by);
        wide_parallel(r.inv.z == 0.0f, a.z, b.y, r.o.z, sz, bz);
    }
    const bool nx = kPar ? r.inv.x < 0.0f : r.neg_x, ny = kPar ? r.inv.y < 0.0f : r.neg_y,
               nz = kPar ? r.inv.z < 0.0f : r.neg_z;
    const float ex = __builtin_fmaf(fabsf(bx), kWideSlack, bx), ey = __builtin_fmaf(fabsf(by), kWideSlack, by),
                ez = __builtin_fmaf(fabsf(bz), kWideSlack, bz);
    const uint32_t lx = __float_as_uint(b.z), ly = __float_as_uint(b.w), lz = __float_as_uint(q.x),
                   hx = __float_as_uint(q.y), hy = __float_as_uint(q.z), hz = __float_as_uint(q.w);
    const uint32_t fx = nx ? hx : lx, gx = nx ? lx : hx, fy = ny ? hy : ly, gy = ny ? ly : hy, fz = nz ? hz : lz,
                   gz = nz ? lz : hz;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        const float ax = __builtin_fmaf(byte_of(fx, k), sx, bx), cx = __builtin_fmaf(byte_of(gx, k), sx, ex);
        const float ay = __builtin_fmaf(byte_of(fy, k), sy, by), cy = __builtin_fmaf(byte_of(gy, k), sy, ey);
        const float az = __builtin_fmaf(byte_of(fz, k), sz, bz), cz = __builtin_fmaf(byte_of(gz, k), sz, ez);
        key[k] = fmaxf(fmaxf(fmaxf(ax, ay), az), r.t_min);
        pass[k] = !(key[k] > fminf(fminf(fminf(cx, cy), cz), t_cull));
    }
}

// Four children in the order of their keys.
__device__ __forceinline__ void wide_sort(float* key, uint32_t* kid) {
    auto order = [&](int i, int j) {
        // loaded first: a select between array elements becomes one between their indexes
        const float ki = key[i], kj = key[j];
        const uint32_t ri = kid[i], rj = kid[j];
        const bool sw = kj < ki;
        key[i] = sw ? kj : ki;
        key[j] = sw ? ki : kj;
        kid[i] = sw ? rj : ri;
        kid[j] = sw ? ri : rj;
    };
    order(0, 1);
    order(2, 3);
    order(0, 2);
    order(1, 3);
    order(1, 2);
}

// Entries of a lane's LDS stack (`stride` words apart, so lanes never share a
// bank). Of 200 000 random rays through 2^20 random triangles 23 held more than
// 16 at once, one more than 20.
constexpr int kWideStack = 20;

// Walks the records from the root, entering boxes up to t_cull (which `leaf`
// may lower), the nearest child first. leaf(at, ref) tests the triangle of one
// leaf child (at = 4 * record + child); true ends the walk (any hit).
// share() runs on every lane after each round of leaf tests; true ends the walk
// of a lane (lanes that walk parts of one ray tell each other); a lane with `skip`
// walks nothing and takes part in that. A lane whose step enters leaf children holds them and does not step again until they
// are tested; the wave tests held leaves together once 1 / kGatherDiv of its
// working lanes hold some, or none can step on. kPar: some lane of the wave has
// an axis-parallel direction. Returns false when the stack overflowed; *bad is
// set on a malformed array (record out of range, a record entered twice).
template <bool kPar, typename Leaf, typename Share>
__device__ __forceinline__ bool wide_walk(const WideNode* __restrict__ wide, uint32_t records, const SlabRay& r,
                                          const float& t_cull, bool skip, uint32_t* stack, int stride,
                                          uint32_t& visits, bool& bad, Leaf&& leaf, Share&& share) {
    uint32_t c = 0, hc = 0, hmask = 0;
    uint4 ref = make_uint4(0, 0, 0, 0);
    int sp = 0;
    uint32_t guard = records;  // each record is entered once
    bool done = skip, overflow = false;
    for (;;) {
        if (!done & (hmask == 0)) {
            if (c >= records || guard-- == 0) {
                bad = true;
                done = true;
            } else {
                float4 a, b, q;
                load_wide(wide, c, a, b, q, ref);
                visits += 2;
                float key[4];
                bool pass[4];
                wide_boxes<kPar>(a, b, q, r, t_cull, key, pass);
                uint32_t kid[4] = {ref.x, ref.y, ref.z, ref.w};
                uint32_t mask = 0;
#pragma unroll
                for (int k = 0; k < 4; ++k) {
                    const bool is_leaf = int32_t(kid[k]) < 0;
                    key[k] = (pass[k] & !is_leaf) ? key[k] : INFINITY;
                    mask |= (pass[k] & is_leaf) ? (1u << k) : 0u;
                }
                hc = c;
                hmask = mask;
                wide_sort(key, kid);
                if (key[0] < INFINITY) {
                    c = kid[0];
                    if (key[1] < INFINITY) {
                        const bool p2 = key[2] < INFINITY, p3 = key[3] < INFINITY;
                        if (sp + 1 + int(p2) + int(p3) > kWideStack) {
                            overflow = true;
                            done = true;
                            hmask = 0;
                        } else {
                            if (p3) stack[sp++ * stride] = kid[3];
                            if (p2) stack[sp++ * stride] = kid[2];
                            stack[sp++ * stride] = kid[1];
                        }
                    }
                } else if (sp == 0) {
                    done = true;
                } else {
                    --sp;
                    c = stack[sp * stride];
                }
            }
        }
        const bool holds = hmask != 0;
        const uint64_t want = __ballot(holds);
        const uint64_t more = __ballot(!done & !holds);
        if (!more) {
            if (!want) break;
        } else if (__popcll(want) * kGatherDiv < __popcll(want | more)) {
            continue;
        }
        while (hmask) {  // each lane's first held leaf, then its second, ...
            const uint32_t k = uint32_t(__ffs(int(hmask))) - 1u;
            hmask &= hmask - 1u;
            const uint32_t r0 = (k & 1u) ? ref.y : ref.x, r1 = (k & 1u) ? ref.w : ref.z;
            if (leaf(4u * hc + k, (k & 2u) ? r1 : r0)) {
                done = true;
                hmask = 0;
            }
        }
        if (share()) done = true;
    }
    return !overflow;
}

// A tree as the ray kernels read it: the right-first preorder node array and the
// four-child records over it.
struct RayTree {
    const lux_bvh_node* nodes;
    const WideNode* wide;
    const int32_t* wide_leaf;
    int32_t node_count;  // 2 n - 1
    uint32_t records;    // n - 1, or 0: the preorder walk only
};

inline RayTree ray_tree(const BvhDev& d) {
    RayTree t;
    t.nodes = d.nodes;
    t.wide = d.wide;
    t.wide_leaf = d.wide_leaf;
    t.node_count = d.n > 0 ? 2 * d.n - 1 : 0;
    t.records = (d.n > 1 && uint32_t(d.n) <= kMaxWideRecords) ? uint32_t(d.n - 1) : 0u;
    return t;
}

// A ray's hit: primitive (-1: none), distance, its leaf's preorder position;
// failed: the preorder walk decides.
struct WideHit {
    int prim = -1;
    int pos = 0;
    float t = 0;
    bool failed = false;
};

// Lanes per ray of a launch over n rays whose walks leave the chip idle: where
// the parts of wide_query pay. Closest hit, 1 / 4 / 8 / 16 lanes: 2^14 rays in
// 2^20 random triangles (with their build) 884 / 648 / 590 / 569 us, 2^15 395 /
// 165 / 123 / 135, 2^16 in 2^18 (with the refit) 431 / 260 / 257 / 283; 2^17 in
// 500 000 382 / 277 / 285, on a sphere mesh 133 / 119 / 122; at 2^18 one lane is
// the best for the soup (422 / 455) and within 6 % on the sphere.
constexpr uint32_t kPartsMaxRays = 1u << 17;
// A walk through a handful of records is no chain worth cutting: 12 triangles, parts /
// one lane a ray, 1000 rays 3.9 / 4.0 us, 2^14 6.5 / 4.5, 2^17 8.9 / 5.5 (sibling
// pairs before: 5.7, 6.1, 47).
constexpr uint32_t kPartsMinRecords = 16;
__host__ __device__ inline int lanes_per_ray(uint32_t n) {
    return n <= (1u << 14) ? 16 : n <= (1u << 16) ? 8 : n <= kPartsMaxRays ? 4 : 1;
}

// Part `part` of `group` of the interval in which ray r meets the root box: lo and
// hi (the ray's bounds before) become its ends. An interval that is empty or not
// finite leaves the whole ray to the first lane; the others get false.
__device__ __forceinline__ bool ray_part(const lux_bvh_node* __restrict__ nodes, const SlabRay& r, int group, int part,
                                         float& lo, float& hi) {
    float4 a, b;
    load_node(nodes, 0, a, b);
    float enter;
    (void)slab_near<true>(r, INFINITY, a.x, a.y, a.z, a.w, b.x, b.y, enter);
    float leave = hi;
    if (!r.par_x) leave = fminf(leave, ((r.neg_x ? a.x : a.w) - r.o.x) * r.inv.x);
    if (!r.par_y) leave = fminf(leave, ((r.neg_y ? a.y : b.x) - r.o.y) * r.inv.y);
    if (!r.par_z) leave = fminf(leave, ((r.neg_z ? a.z : b.y) - r.o.z) * r.inv.z);
    const float step = (leave - enter) / float(group);
    const bool cut = step > 0.0f && step < 1e30f;
    if (cut && part + 1 < group) hi = enter + step * float(part + 1);
    if (cut && part != 0) lo = enter + step * float(part);
    return cut || part == 0;
}

// One ray, on `group` lanes in a row (a power of two; 1: a lane by itself), this
// lane walking part `part` of the interval in which the ray meets the root box.
// Every lane of a group has the same ray and gets the group's result. any: any
// hit in (t_min, t_max), otherwise the closest; `ignore` is a primitive to pass
// over (-1: none).
// A launch that leaves most of the chip idle lasts as long as its longest walk, a
// chain of dependent loads; parts cut the chain (2^20 random triangles, 2^14
// random rays: 330 records for the longest ray, 148 in 4 parts, 87 in 8) for more
// records in all (50, 130 and 194 a ray). A box met by the ray in [t_min, t_max]
// is met in some part, so every triangle the whole walk tests is tested by some
// lane; the hit is the smallest (t, preorder position) over the lanes, as it is
// over one lane's walk. With t_max fixed, whether a leaf's box passes does not
// depend on the visit order, so an any-hit walk may end at any triangle hit in a
// leaf whose own box passes; near child first meets one soon.
// kOwnIds: see preorder_query.
template <bool kOwnIds = false>
__device__ __forceinline__ WideHit wide_query(const RayTree& tree, const lux_triangle* __restrict__ tris,
                                              int tri_count, const f3& o, const f3& d, float t_min, float t_bound,
                                              bool any, int ignore, int group, int part, uint32_t* stack, int stride,
                                              DevInfo* info, uint32_t& visits, uint32_t& tests) {
    WideHit hit;
    if (tree.records == 0 || !wide_takes(d)) {
        hit.failed = true;
        return hit;
    }
    SlabRay sr = make_slab_ray(o, d, t_min);
    float hi = t_bound;
    const bool skip = group > 1 && !ray_part(tree.nodes, sr, group, part, sr.t_min, hi);
    float t_max = t_bound;  // the held bound
    float t_cull = wide_bound(hi);
    int best = -1;
    uint32_t best_at = 0;
    bool bad = false, bad_prim = false;
    auto leaf = [&](uint32_t at, uint32_t ref) {
        const uint32_t prim = ref & kIndexMask;
        if (int(prim) == ignore) return false;
        if (prim >= uint32_t(tri_count)) {  // no child, or a leaf id out of range
            bad_prim |= ref != kWideEmpty || (!kOwnIds && tree.wide_leaf[at] >= 0);
            return false;
        }
        const float* p = reinterpret_cast<const float*>(tris + prim);
        ++tests;
        float t, u, v;
        if (!tri_uvt(o, d, make3(p[0], p[1], p[2]), make3(p[3], p[4], p[5]), make3(p[6], p[7], p[8]), t, u, v) ||
            !(t > t_min))
            return false;
        if (t < t_max || (!any && best >= 0 && t == t_max && tree.wide_leaf[at] < tree.wide_leaf[best_at])) {
            best = int(prim);
            best_at = at;
            if (any) return true;
            t_max = t;
            t_cull = fminf(t_cull, t + fabsf(t) * kSoftWindow);
        }
        return false;
    };
    auto share = [&]() {
        if (group == 1) return false;
        float t = best < 0 ? INFINITY : any ? -INFINITY : t_max;
        for (int off = 1; off < group; off <<= 1) t = fminf(t, __shfl_xor(t, off, 64));
        if (any) return t < INFINITY;
        t_cull = fminf(t_cull, t + fabsf(t) * kSoftWindow);
        return false;
    };
    hit.failed = wave_any_parallel(sr)
                     ? !wide_walk<true>(tree.wide, tree.records, sr, t_cull, skip, stack, stride, visits, bad, leaf, share)
                     : !wide_walk<false>(tree.wide, tree.records, sr, t_cull, skip, stack, stride, visits, bad, leaf, share);
    if (kOwnIds && bad_prim) set_error(info, kErrPrimRange);
    if (bad) set_error(info, kErrWalkOrder);
    if (!kOwnIds) hit.failed |= bad_prim;  // the leaf's own box decides
    hit.prim = best;
    hit.t = t_max;
    if (best >= 0) hit.pos = tree.wide_leaf[best_at];
    if (group > 1) {
        // the smallest (t, position) of the group, on every lane
        int fail = hit.failed;
        for (int off = 1; off < group; off <<= 1) {
            const float ot = __shfl_xor(hit.t, off, 64);
            const int op = __shfl_xor(hit.pos, off, 64), oid = __shfl_xor(hit.prim, off, 64);
            fail |= __shfl_xor(fail, off, 64);
            const bool before = (!any && ot != hit.t) ? ot < hit.t : op < hit.pos;
            if (oid >= 0 && (hit.prim < 0 || before)) {
                hit.t = ot;
                hit.pos = op;
                hit.prim = oid;
            }
        }
        hit.failed = fail != 0;
    }
    if (!hit.failed && hit.prim >= 0) {
        sr.t_min = t_min;
        hit.failed = !wide_settled(tree.nodes, tree.node_count, hit.pos, sr, hit.t, info);
    }
    return hit;
}

// Right-first preorder walk: the rays that wide_query hands back, one-leaf trees
// and trees beyond 32-bit record offsets. any: stop at the first accepted
// triangle. visits counts node loads, tests triangle tests.
// A leaf id at or above tri_count is an error for a ray that meets the leaf's box no
// farther than its hit (an any-hit query: that finds none), in whatever order: a walk
// that passed such a leaf is made again up to the hit (kOwnIds: ids the library gave
// itself, an error at once).
template <bool kOwnIds = false>
__device__ __forceinline__ WideHit preorder_query(const RayTree& tree, const lux_triangle* __restrict__ tris,
                                                  int tri_count, const f3& o, const f3& d, float t_min,
                                                  float t_bound, bool any, int ignore, DevInfo* info,
                                                  uint32_t& visits, uint32_t& tests) {
    const SlabRay sr = make_slab_ray(o, d, t_min);
    WideHit hit;
    hit.t = t_bound;
    bool bad_order = false;
    for (bool again = false;; again = true) {
        int k = 0;
        bool bad_prim = false;
        while (uint32_t(k) < uint32_t(tree.node_count)) {
            float4 a, b;
            load_node(tree.nodes, k, a, b);
            ++visits;
            const int prim = __float_as_int(b.z);
            const bool pass = slab_hit(sr, hit.t, a.x, a.y, a.z, a.w, b.x, b.y);
            int next = (pass && prim < 0) ? k + 1 : __float_as_int(b.w);
            const bool test = pass && prim >= 0 && prim != ignore;
            bad_prim |= test && prim >= tri_count;
            if (test && prim < tri_count) {
                const float* p = reinterpret_cast<const float*>(tris + prim);
                ++tests;
                float t, u, v;
                if (tri_hit(o, d, t_min, hit.t, make3(p[0], p[1], p[2]), make3(p[3], p[4], p[5]),
                            make3(p[6], p[7], p[8]), t, u, v)) {
                    hit.prim = prim;
                    hit.t = t;
                    if (any) next = -1;  // done
                }
            }
            if (next >= 0 && next <= k) {  // preorder positions only grow
                bad_order = true;
                break;
            }
            k = next;
        }
        if (!bad_prim || (any && hit.prim >= 0 && !kOwnIds)) break;
        if (kOwnIds || again || hit.prim < 0) {
            set_error(info, kErrPrimRange);
            break;
        }
    }
    if (bad_order) set_error(info, kErrWalkOrder);
    return hit;
}

}  // namespace lux
