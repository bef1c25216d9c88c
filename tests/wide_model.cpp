// wide_model.cpp -- the library's four-child records and their walk
// (lux_amd/csrc/wide.hpp, as it stands) on the CPU, a wave of 64 lanes at a time.
#include "wide.hpp"

using namespace lux;

extern "C" {

// Records of a tree given as radix tree links (bit 31: leaf), preorder positions
// and stackless nodes.
uint32_t wide_fill(int n, const uint32_t* left, const uint32_t* right, const int32_t* pre_internal,
                   const int32_t* pre_leaf, const lux_bvh_node* nodes, WideNode* wide, int32_t* wide_leaf) {
    DevInfo info{};
    for (int i = 0; i < n - 1; ++i)
        fill_wide(n, i, left, right, pre_internal, pre_leaf, nodes, wide, wide_leaf, &info);
    return info.error;
}

// Rays on `group` lanes each, as the query kernels trace them: the records' walk,
// then the preorder walk for the rays it hands back (counted in *again). Returns
// the error bits.
uint32_t wide_trace(int n, const lux_bvh_node* nodes, const WideNode* wide, const int32_t* wide_leaf,
                    const lux_triangle* tris, int tri_count, const lux_ray* rays, int count, int any, int group,
                    int32_t* ids, float* t, int32_t* again) {
    DevInfo info{};
    RayTree tree{nodes, wide, wide_leaf, 2 * n - 1, uint32_t(n - 1)};
    *again = 0;
    const int per = simt::kLanes / group;
    uint32_t stack[kWideStack * simt::kLanes];
    for (int first = 0; first < count; first += per) {
        const int here = count - first < per ? count - first : per;
        simt::run(here * group, [&](int lane) {
            const int i = first + lane / group, part = lane % group;
            const lux_ray& r = rays[i];
            const f3 o = ld3(r.origin), d = ld3(r.direction);
            uint32_t visits = 0, tests = 0;
            WideHit h = wide_query(tree, tris, tri_count, o, d, r.t_min, r.t_max, any != 0, -1, group, part,
                                   stack + lane, simt::kLanes, &info, visits, tests);
            if (h.failed && part == 0) {
                ++*again;
                h = preorder_query(tree, tris, tri_count, o, d, r.t_min, r.t_max, any != 0, -1, &info, visits, tests);
            }
            if (part == 0) {
                ids[i] = h.prim;
                t[i] = h.prim >= 0 ? h.t : INFINITY;
            }
        });
    }
    return info.error;
}
}
