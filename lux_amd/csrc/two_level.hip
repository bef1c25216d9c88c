// two_level.hip -- builds two-level (instanced) scenes and launches their walk
// (two_level.hpp) over ray arrays.
#include <algorithm>
#include <cmath>
#include <cstring>

#include "two_level.hpp"

namespace lux {
namespace {

constexpr int kBlock = 128;
// Rays are walked in ray order from this many rays and mesh triangles on: below,
// the meshes' records and triangles (112 bytes each) come out of the L2s (4 MiB per
// XCD) or the sort costs more than it gives. Closest hit over 50 or 64 instances,
// sorted (sort included) / in input order: 262 144 triangles 1.45 / 1.27 ms at
// 300 000 rays, 1.36 / 1.48 at 600 000, 2.04 / 2.84 at 2^20; 131 072 triangles 1.64
// / 1.62 at 2^20 rays; 60 000 triangles 4.37 / 4.22 at 2^22.
constexpr int kTwoLevelOrderMinRays = 1 << 19;
constexpr int kTwoLevelOrderMinTris = 1 << 18;

__device__ __forceinline__ lux_scene_hit scene_hit(const TwoLevelHit& h) {
    lux_scene_hit out;
    out.primitive_id = h.prim;
    out.t = h.prim >= 0 ? h.t : INFINITY;
    out.u = h.prim >= 0 ? h.u : 0.0f;
    out.v = h.prim >= 0 ? h.v : 0.0f;
    out.instance_id = h.instance;
    out.local_primitive_id = h.local;
    return out;
}

// One ray: the records' walk, or the preorder walk where it cannot settle the ray.
template <bool kAny>
__device__ __forceinline__ TwoLevelHit query(const TwoLevelView& s, const lux_ray* __restrict__ rays, int i,
                                             const int32_t* __restrict__ ignore, int group, int part,
                                             uint32_t* stack) {
    const float t_min = rays[i].t_min, t_max = rays[i].t_max;
    const int ign = ignore ? ignore[i] : -1;
    auto world = [&](f3& o, f3& d) {
        o = ld3(rays[i].origin);
        d = ld3(rays[i].direction);
    };
    TwoLevelHit h;
    if (!two_level_wide<false>(s, world, t_min, __builtin_canonicalizef(t_max), kAny, ign, group, part, stack, kBlock,
                               h))
        h = two_level_walk(s, world, t_min, t_max, kAny, ign);
    return h;
}

// `group` lanes walk one ray (lanes_per_ray).
// 7 waves per SIMD (72 VGPRs): 2^20 rays over 64 instances 2.10 / 2.02 / 2.36 ms
// at 6 / 7 / 8.
// `order`: the rays in ray order (a permutation of [0, n)), or null for input
// order; a result lands at its ray's own index: a lux_scene_hit, or one byte (kAny).
template <bool kAny>
__global__ __launch_bounds__(kBlock) __attribute__((amdgpu_waves_per_eu(7))) void k_two_level(
    TwoLevelView s, const uint32_t* __restrict__ order, const lux_ray* __restrict__ rays,
    const int32_t* __restrict__ ignore, int n, int group, void* __restrict__ out) {
    const uint32_t lane = xcd_block() * kBlock + threadIdx.x;
    const int j = int(lane / uint32_t(group)), part = int(lane & uint32_t(group - 1));
    if (j >= n) return;
    __shared__ uint32_t stack[kWideStack * kBlock];
    const int i = order ? int(order[j]) : j;
    if (uint32_t(i) >= uint32_t(n)) {  // only if the sort itself reported an error
        set_error(s.info, kErrSpinLimit);
        return;
    }
    const TwoLevelHit h = query<kAny>(s, rays, i, ignore, group, part, stack + threadIdx.x);
    if (part != 0) return;
    if (kAny)
        static_cast<uint8_t*>(out)[i] = h.prim >= 0 ? 1 : 0;
    else
        static_cast<lux_scene_hit*>(out)[i] = scene_hit(h);
}

template <typename T>
T* dalloc_n(size_t count) {
    void* p = nullptr;
    hipError_t e = hipMalloc(&p, std::max<size_t>(count, 1) * sizeof(T));
    if (e != hipSuccess) throw Error(LUX_ERR_OUT_OF_MEMORY, std::string("hipMalloc failed: ") + hipGetErrorString(e));
    return static_cast<T*>(p);
}

bool box_is_empty(const lux_aabb& b) {
    return b.p_min.x > b.p_max.x || b.p_min.y > b.p_max.y || b.p_min.z > b.p_max.z;
}

// det3 and the affine test of src/core/mat4.cuh:86-104, host side.
float affine_det3(const float* m) {
    return m[0] * (m[5] * m[10] - m[6] * m[9]) - m[1] * (m[4] * m[10] - m[6] * m[8]) +
           m[2] * (m[4] * m[9] - m[5] * m[8]);
}
bool affine_invertible(const float* m) {
    return std::fabs(m[12]) <= 1e-6f && std::fabs(m[13]) <= 1e-6f && std::fabs(m[14]) <= 1e-6f &&
           std::fabs(m[15] - 1.0f) <= 1e-6f && std::fabs(affine_det3(m)) > 1e-12f;
}
bool product_near_identity(const float* a, const float* b) {
    for (int i = 0; i < 4; ++i)
        for (int j = 0; j < 4; ++j) {
            float s = 0.0f;
            for (int k = 0; k < 4; ++k) s += a[4 * i + k] * b[4 * k + j];
            if (!(std::fabs(s - (i == j ? 1.0f : 0.0f)) <= 1e-4f)) return false;
        }
    return true;
}

void validate_instances(const lux_instance* instances, int count, int mesh_count) {
    if (count < 0) throw Error(LUX_ERR_INVALID_ARGUMENT, "negative instance count");
    if (count > 0 && !instances) throw Error(LUX_ERR_INVALID_ARGUMENT, "null instance array");
    for (int i = 0; i < count; ++i) {
        const lux_instance& in = instances[i];
        if (in.mesh_id < 0 || in.mesh_id >= mesh_count)
            throw Error(LUX_ERR_INVALID_ARGUMENT, "instance " + std::to_string(i) + ": mesh id out of range");
        if (!instance_transform_valid(in.object_to_world, in.world_to_object))
            throw Error(LUX_ERR_INVALID_ARGUMENT,
                        "instance " + std::to_string(i) + ": transform must be affine-invertible with a consistent inverse");
    }
}

void sync_and_check(const BvhDev& d, hipStream_t stream, const char* what) {
    uint32_t error = 0;
    if (d.info)
        hip_check(hipMemcpyAsync(&error, &d.info->error, sizeof(error), hipMemcpyDeviceToHost, stream),
                  "read device errors");
    hip_check(hipStreamSynchronize(stream), what);
    if (error != 0) throw Error(LUX_ERR_DEVICE_CHECK, std::string("device check failed in ") + what);
}

// The records over the TLAS with its culling boxes (TwoLevelDev::tlas), and
// each instance's leaf position: a node array of the TLAS's topology, each leaf
// box the instance's world bounds intersected with the world box of its mesh's
// bounding sphere (both widened as below), each internal box the union of its two
// children. Every box still holds every world-space ray point that can hit the
// geometry below it, so only the culling changes.
// `nodes` (n > 0 instances, filled here) has to last until the stream is waited for.
void build_tlas_wide(TwoLevelDev& s, const lux_instance* instances, std::vector<DevInstance>& rec,
                     std::vector<lux_bvh_node>& nodes, hipStream_t stream) {
    const int n = s.tlas.n;
    const int count = 2 * n - 1;
    nodes.resize(static_cast<size_t>(count));
    hip_check(hipMemcpyAsync(nodes.data(), s.tlas.nodes, sizeof(lux_bvh_node) * count, hipMemcpyDeviceToHost, stream),
              "D2H TLAS");
    sync_and_check(s.tlas, stream, "TLAS build");
    // A leaf box must hold every world point w(t) of a ray whose object-space
    // image p(t) = inv w(t) lies in the mesh: M p(t) = (M inv) w(t) lies in the
    // transformed mesh, and M inv is the identity only to the scene
    // validation's 1e-4 per entry, so w(t) may sit up to 3 e |w| + e_t off it
    // (e, e_t: the largest deviation of M inv from the identity in the 3x3 and
    // translation parts). Both boxes are widened by that, plus a margin for
    // float rounding, before they are intersected.
    auto leaf_box = [&](int inst) {
        const lux_instance& in = instances[inst];
        const float* m = in.object_to_world;
        const float* v = in.world_to_object;
        double e3 = 0, et = 0;
        for (int r = 0; r < 3; ++r)
            for (int c = 0; c < 4; ++c) {
                double x = c == 3 ? double(m[4 * r + 3]) : 0.0;
                for (int k = 0; k < 3; ++k) x += double(m[4 * r + k]) * v[4 * k + c];
                if (c == 3) {
                    et = std::max(et, std::fabs(x));
                } else {
                    e3 = std::max(e3, std::fabs(x - (r == c ? 1.0 : 0.0)));
                }
            }
        const lux_aabb& ref = in.world_bounds;
        const double R = std::max({std::fabs(double(ref.p_min.x)), std::fabs(double(ref.p_min.y)),
                                   std::fabs(double(ref.p_min.z)), std::fabs(double(ref.p_max.x)),
                                   std::fabs(double(ref.p_max.y)), std::fabs(double(ref.p_max.z))});
        const double pad = 3.0 * e3 * R + et + 1e-5 * (R + 1e-30);
        double lo[3] = {ref.p_min.x - pad, ref.p_min.y - pad, ref.p_min.z - pad};
        double hi[3] = {ref.p_max.x + pad, ref.p_max.y + pad, ref.p_max.z + pad};
        const float* sph = &s.mesh_sphere[4 * size_t(in.mesh_id)];
        if (sph[3] >= 0) {
            for (int r = 0; r < 3; ++r) {
                const double c = double(m[4 * r]) * sph[0] + double(m[4 * r + 1]) * sph[1] +
                                 double(m[4 * r + 2]) * sph[2] + double(m[4 * r + 3]);
                const double h = double(sph[3]) * std::sqrt(double(m[4 * r]) * m[4 * r] +
                                                            double(m[4 * r + 1]) * m[4 * r + 1] +
                                                            double(m[4 * r + 2]) * m[4 * r + 2]);
                lo[r] = std::max(lo[r], c - h - pad);
                hi[r] = std::min(hi[r], c + h + pad);
            }
        }
        lux_aabb b;
        b.p_min = lux_vec3{float(lo[0]), float(lo[1]), float(lo[2])};
        b.p_max = lux_vec3{float(hi[0]), float(hi[1]), float(hi[2])};
        // rounding to float must not move a face inward
        b.p_min = lux_vec3{std::nextafter(b.p_min.x, -INFINITY), std::nextafter(b.p_min.y, -INFINITY),
                           std::nextafter(b.p_min.z, -INFINITY)};
        b.p_max = lux_vec3{std::nextafter(b.p_max.x, INFINITY), std::nextafter(b.p_max.y, INFINITY),
                           std::nextafter(b.p_max.z, INFINITY)};
        return b;
    };
    // children have larger preorder positions than their parent: the right child
    // is the next node, the left child the right one's escape
    for (int k = count - 1; k >= 0; --k) {
        lux_bvh_node& nd = nodes[size_t(k)];
        if (nd.primitive_id >= 0) {
            if (nd.primitive_id < s.instance_count) {
                rec[size_t(nd.primitive_id)].tlas_pos = k;
                nd.bounds = leaf_box(nd.primitive_id);
            }
            continue;
        }
        const int left = k + 1 < count ? nodes[size_t(k) + 1].escape : -1;
        if (left <= k + 1 || left >= count) throw Error(LUX_ERR_DEVICE_CHECK, "malformed TLAS node array");
        const lux_aabb& l = nodes[size_t(left)].bounds;
        const lux_aabb& r = nodes[size_t(k) + 1].bounds;
        nd.bounds.p_min = lux_vec3{std::min(l.p_min.x, r.p_min.x), std::min(l.p_min.y, r.p_min.y),
                                   std::min(l.p_min.z, r.p_min.z)};
        nd.bounds.p_max = lux_vec3{std::max(l.p_max.x, r.p_max.x), std::max(l.p_max.y, r.p_max.y),
                                   std::max(l.p_max.z, r.p_max.z)};
    }
    if (n < 2) return;
    if (s.tlas_cull_capacity < count) {
        if (s.tlas_cull) hip_check(hipFree(s.tlas_cull), "hipFree culling nodes");
        s.tlas_cull = nullptr;
        s.tlas_cull_capacity = 0;
        s.tlas_cull = dalloc_n<lux_bvh_node>(size_t(count));
        s.tlas_cull_capacity = count;
    }
    hip_check(hipMemcpyAsync(s.tlas_cull, nodes.data(), sizeof(lux_bvh_node) * count, hipMemcpyHostToDevice, stream),
              "H2D culling TLAS");
    wide_from(s.tlas, s.tlas_cull, s.tlas.wide, s.tlas.wide_leaf, stream);
}

// TLAS over the non-empty world bounds (ids = instance ids) and the instance
// records; first ordinals follow the instances in order (each adds its mesh's
// triangle count).
void upload_instances(TwoLevelDev& s, const lux_instance* instances, int count, hipStream_t stream) {
    std::vector<DevInstance> rec(static_cast<size_t>(std::max(count, 0)));
    std::vector<lux_aabb> boxes;
    std::vector<int32_t> ids;
    int64_t cursor = 0;
    for (int i = 0; i < count; ++i) {
        const lux_instance& in = instances[i];
        DevInstance& r = rec[i];
        std::memcpy(r.inv, in.world_to_object, sizeof(r.inv));
        r.mesh = in.mesh_id;
        const int64_t tri = s.mesh_tri_off[in.mesh_id + 1] - s.mesh_tri_off[in.mesh_id];
        if (cursor + tri > INT32_MAX) throw Error(LUX_ERR_INVALID_ARGUMENT, "more than 2^31 scene primitives");
        r.first = int32_t(cursor);
        r.wide = s.blas[in.mesh_id].wide;
        r.tris = s.soup + s.mesh_tri_off[in.mesh_id];
        r.tri_count = int32_t(tri);
        r.tlas_pos = -1;
        cursor += tri;
        if (box_is_empty(in.world_bounds)) continue;
        boxes.push_back(in.world_bounds);
        ids.push_back(i);
    }
    const int n = int(boxes.size());
    s.whole = false;
    s.host_instances.assign(instances, instances + count);
    s.instance_count = count;
    s.scene_primitives = cursor;
    s.tlas_instances = n;
    s.tlas.holds = kCopyRecords;  // the culling records
    bvh_allocate(s.tlas, n, stream);
    if (n > 0) {
        hip_check(hipMemcpyAsync(s.tlas.boxes, boxes.data(), sizeof(lux_aabb) * n, hipMemcpyHostToDevice, stream),
                  "H2D world bounds");
        hip_check(hipMemcpyAsync(s.tlas.ids, ids.data(), sizeof(int32_t) * n, hipMemcpyHostToDevice, stream),
                  "H2D instance ids");
    }
    lbvh_build(s.tlas, s.tlas.boxes, s.tlas.ids, n, stream);
    uint64_t limit = n > 1 ? 2u * uint64_t(n) : uint64_t(n);
    for (int i = 0; i < count; ++i) {
        const int tri = s.mesh_tri_off[instances[i].mesh_id + 1] - s.mesh_tri_off[instances[i].mesh_id];
        limit += tri > 1 ? 2u * uint64_t(tri) : uint64_t(tri);
    }
    s.step_limit = uint32_t(std::min<uint64_t>(limit + 1, 0xffffffffu));
    std::vector<lux_bvh_node> nodes;
    if (n > 0) build_tlas_wide(s, instances, rec, nodes, stream);
    if (s.instance_capacity < count || !s.instances) {
        if (s.instances) hip_check(hipFree(s.instances), "hipFree instances");
        s.instances = nullptr;
        s.instance_capacity = 0;
        s.instances = dalloc_n<DevInstance>(rec.size());
        s.instance_capacity = count;
    }
    if (!rec.empty())
        hip_check(hipMemcpyAsync(s.instances, rec.data(), sizeof(DevInstance) * rec.size(), hipMemcpyHostToDevice,
                                 stream),
                  "H2D instances");
    sync_and_check(s.tlas, stream, "TLAS records");
    s.whole = true;
}

}  // namespace

bool instance_transform_valid(const float* m16, const float* inv16) {
    return affine_invertible(m16) && affine_invertible(inv16) && product_near_identity(m16, inv16) &&
           product_near_identity(inv16, m16);
}

void inverse_affine(const float* m, float* r) {
    for (int i = 0; i < 16; ++i) r[i] = (i % 5 == 0) ? 1.0f : 0.0f;
    const float a00 = m[0], a01 = m[1], a02 = m[2];
    const float a10 = m[4], a11 = m[5], a12 = m[6];
    const float a20 = m[8], a21 = m[9], a22 = m[10];
    const float det = affine_det3(m);
    if (std::fabs(det) <= 1e-12f) return;
    const float inv_det = 1.0f / det;
    r[0] = (a11 * a22 - a12 * a21) * inv_det;
    r[1] = -(a01 * a22 - a02 * a21) * inv_det;
    r[2] = (a01 * a12 - a02 * a11) * inv_det;
    r[4] = -(a10 * a22 - a12 * a20) * inv_det;
    r[5] = (a00 * a22 - a02 * a20) * inv_det;
    r[6] = -(a00 * a12 - a02 * a10) * inv_det;
    r[8] = (a10 * a21 - a11 * a20) * inv_det;
    r[9] = -(a00 * a21 - a01 * a20) * inv_det;
    r[10] = (a00 * a11 - a01 * a10) * inv_det;
    const float tx = m[3], ty = m[7], tz = m[11];
    r[3] = -(r[0] * tx + r[1] * ty + r[2] * tz);
    r[7] = -(r[4] * tx + r[5] * ty + r[6] * tz);
    r[11] = -(r[8] * tx + r[9] * ty + r[10] * tz);
    r[12] = r[13] = r[14] = 0.0f;
    r[15] = 1.0f;
}

lux_aabb transform_bounds(const float* m, const lux_aabb& b) {
    lux_aabb r;
    r.p_min = lux_vec3{INFINITY, INFINITY, INFINITY};
    r.p_max = lux_vec3{-INFINITY, -INFINITY, -INFINITY};
    if (box_is_empty(b)) return r;
    for (int z = 0; z <= 1; ++z)
        for (int y = 0; y <= 1; ++y)
            for (int x = 0; x <= 1; ++x) {
                const float cx = x ? b.p_max.x : b.p_min.x, cy = y ? b.p_max.y : b.p_min.y,
                            cz = z ? b.p_max.z : b.p_min.z;
                float px = m[0] * cx + m[1] * cy + m[2] * cz + m[3];
                float py = m[4] * cx + m[5] * cy + m[6] * cz + m[7];
                float pz = m[8] * cx + m[9] * cy + m[10] * cz + m[11];
                const float w = m[12] * cx + m[13] * cy + m[14] * cz + m[15];
                if (w != 1.0f) {
                    px = px / w;
                    py = py / w;
                    pz = pz / w;
                }
                r.p_min = lux_vec3{std::fmin(r.p_min.x, px), std::fmin(r.p_min.y, py), std::fmin(r.p_min.z, pz)};
                r.p_max = lux_vec3{std::fmax(r.p_max.x, px), std::fmax(r.p_max.y, py), std::fmax(r.p_max.z, pz)};
            }
    return r;
}

void two_level_release(TwoLevelDev& s) {
    for (BvhDev& b : s.blas) bvh_release(b);
    bvh_release(s.tlas);
    void* ptrs[] = {s.soup, s.meshes, s.instances, s.tlas_cull};
    for (void* p : ptrs)
        if (p) (void)hipFree(p);
    s = TwoLevelDev{};
}

void two_level_build(TwoLevelDev& s, const lux_triangle* tris, const int32_t* offsets, int mesh_count,
                     const lux_instance* instances, int instance_count, hipStream_t stream) {
    if (mesh_count < 0) throw Error(LUX_ERR_INVALID_ARGUMENT, "negative mesh count");
    if (mesh_count > 0 && !offsets) throw Error(LUX_ERR_INVALID_ARGUMENT, "null mesh offsets");
    if (mesh_count > 0 && offsets[0] != 0) throw Error(LUX_ERR_INVALID_ARGUMENT, "mesh_offsets[0] must be 0");
    for (int m = 0; m < mesh_count; ++m)
        if (offsets[m + 1] < offsets[m]) throw Error(LUX_ERR_INVALID_ARGUMENT, "mesh offsets must not decrease");
    const int total = mesh_count > 0 ? offsets[mesh_count] : 0;
    if (total > 0 && !tris) throw Error(LUX_ERR_INVALID_ARGUMENT, "null triangle array");
    validate_instances(instances, instance_count, mesh_count);
    two_level_release(s);
    s.mesh_count = mesh_count;
    s.mesh_tri_off.assign(size_t(mesh_count) + 1, 0);
    for (int m = 0; m <= mesh_count; ++m) s.mesh_tri_off[m] = mesh_count > 0 ? offsets[m] : 0;
    s.soup = dalloc_n<lux_triangle>(size_t(std::max(total, 1)));
    if (total > 0)
        hip_check(hipMemcpyAsync(s.soup, tris, sizeof(lux_triangle) * total, hipMemcpyHostToDevice, stream),
                  "H2D mesh triangles");
    s.blas.resize(size_t(mesh_count));
    std::vector<DevMesh> meshes(static_cast<size_t>(mesh_count));
    for (int m = 0; m < mesh_count; ++m) {
        const int n = offsets[m + 1] - offsets[m];
        s.blas[m].holds = kCopyRecords;
        // BLAS input (triangle_bounds, local ids) computed on the device from
        // the soup copied above
        lbvh_build_triangles(s.blas[m], s.soup + offsets[m], nullptr, nullptr, 0, n, stream);
        tree_copies(s.blas[m], kCopyRecords, stream);
        sync_and_check(s.blas[m], stream, "BLAS build");
        meshes[m].nodes = s.blas[m].nodes;
        meshes[m].wide_leaf = s.blas[m].wide_leaf;
        meshes[m].tris = s.soup + offsets[m];
        meshes[m].node_count = n > 0 ? 2 * n - 1 : 0;
        meshes[m].tri_count = n;
        s.device_bytes += bvh_device_bytes(n, kCopyRecords);
    }
    // each mesh's bounding sphere: the center of its box, the largest vertex
    // distance from it (in double, padded), radius -1 for an empty mesh
    s.mesh_sphere.assign(4 * size_t(mesh_count), 0.0f);
    for (int m = 0; m < mesh_count; ++m) {
        float* sph = &s.mesh_sphere[4 * size_t(m)];
        if (offsets[m + 1] == offsets[m]) {
            sph[3] = -1.0f;
            continue;
        }
        float lo[3] = {INFINITY, INFINITY, INFINITY}, hi[3] = {-INFINITY, -INFINITY, -INFINITY};
        for (int t = offsets[m]; t < offsets[m + 1]; ++t)
            for (const lux_vec3& v : {tris[t].v0, tris[t].v1, tris[t].v2}) {
                const float q[3] = {v.x, v.y, v.z};
                for (int a = 0; a < 3; ++a) {
                    lo[a] = std::min(lo[a], q[a]);
                    hi[a] = std::max(hi[a], q[a]);
                }
            }
        double r2 = 0;
        for (int a = 0; a < 3; ++a) sph[a] = 0.5f * (lo[a] + hi[a]);
        for (int t = offsets[m]; t < offsets[m + 1]; ++t)
            for (const lux_vec3& v : {tris[t].v0, tris[t].v1, tris[t].v2}) {
                const double dx = double(v.x) - sph[0], dy = double(v.y) - sph[1], dz = double(v.z) - sph[2];
                r2 = std::max(r2, dx * dx + dy * dy + dz * dz);
            }
        sph[3] = float(std::sqrt(r2) * (1.0 + 1e-6)) + 1e-30f;
    }
    s.meshes = dalloc_n<DevMesh>(meshes.size());
    if (!meshes.empty())
        hip_check(hipMemcpyAsync(s.meshes, meshes.data(), sizeof(DevMesh) * meshes.size(), hipMemcpyHostToDevice,
                                 stream),
                  "H2D meshes");
    upload_instances(s, instances, instance_count, stream);
    s.device_bytes += sizeof(lux_triangle) * size_t(total) + sizeof(DevMesh) * meshes.size() +
                      sizeof(DevInstance) * size_t(instance_count) + bvh_device_bytes(s.tlas_instances, kCopyRecords) +
                      sizeof(lux_bvh_node) * size_t(std::max(2 * s.tlas_instances - 1, 0));
}

void two_level_set_instances(TwoLevelDev& s, const lux_instance* instances, int instance_count,
                             hipStream_t stream) {
    if (instance_count != s.instance_count)
        throw Error(LUX_ERR_MISMATCH, "instance count differs from the built scene");
    validate_instances(instances, instance_count, s.mesh_count);
    upload_instances(s, instances, instance_count, stream);
}

TwoLevelView two_level_view(const TwoLevelDev& s) {
    if (!s.whole) throw Error(LUX_ERR_INVALID_ARGUMENT, "instances were lost in a failed update: set them again");
    TwoLevelView v;
    v.tlas_nodes = s.tlas.nodes;
    v.tlas_wide = s.tlas.wide;
    v.tlas_records = s.tlas.n > 1 ? uint32_t(s.tlas.n - 1) : 0u;
    v.instances = s.instances;
    v.meshes = s.meshes;
    v.info = s.tlas.info;
    v.tlas_node_count = s.tlas.n > 0 ? 2 * s.tlas.n - 1 : 0;
    v.instance_count = s.instance_count;
    v.mesh_count = s.mesh_count;
    v.step_limit = s.step_limit;
    return v;
}

const uint32_t* two_level_order(RaySortDev& r, const TwoLevelDev& s, const lux_ray* rays, int n, hipStream_t stream) {
    if (s.tlas.n < 1 || n < kTwoLevelOrderMinRays || s.mesh_tri_off.back() < kTwoLevelOrderMinTris) return nullptr;
    return ray_order(r, s.tlas, rays, n, stream);  // origins quantised in the TLAS root box
}

void two_level_closest(const TwoLevelView& v, const uint32_t* order, const lux_ray* rays, const int32_t* ignore,
                       int n, lux_scene_hit* hits, hipStream_t stream) {
    if (n <= 0) return;
    const int group = lanes_per_ray(uint32_t(n));
    LUX_LAUNCH("two_level_closest", k_two_level<false>, div_up(int64_t(n) * group, kBlock), kBlock, 0, stream, v, order,
               rays, ignore, n, group, static_cast<void*>(hits));
}

void two_level_occluded(const TwoLevelView& v, const uint32_t* order, const lux_ray* rays, const int32_t* ignore,
                        int n, uint8_t* occluded, hipStream_t stream) {
    if (n <= 0) return;
    const int group = lanes_per_ray(uint32_t(n));
    LUX_LAUNCH("two_level_occluded", k_two_level<true>, div_up(int64_t(n) * group, kBlock), kBlock, 0, stream, v, order,
               rays, ignore, n, group, static_cast<void*>(occluded));
}

}  // namespace lux
