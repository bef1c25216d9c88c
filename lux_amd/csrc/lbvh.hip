// lbvh.hip -- LBVH construction and refit for gfx950.
//
// Build pipeline (one stream, no host round trip):
//   root_partials  grid-stride min/max of the input boxes (+ id range) into
//                  per-block partials; block 0 clears the histogram
//   morton_hist    every block folds the partials into the root box, then
//                  30-bit Morton codes, identity payload and the four 8-bit
//                  digit histograms
//   sort_pass x4   stable LSD radix pass with decoupled look-back (one read and
//                  one write of key+value per pass)
//   karras         radix tree over the sorted codes (merged 64-bit keys)
//   top_layout     right-first preorder positions of the nodes whose leaf
//                  range spans more than one leaf block, and the right steps
//                  from the "frontier" (local nodes under them) to the root
//   local          one workgroup per block of kLocalLeaves sorted leaves: places
//                  the leaves and the nodes inside the block, unions boxes
//                  bottom-up inside the block with LDS arrival counters, and
//                  leaves prefix / suffix unions of the block's frontier nodes
//   top_boxes      one wave per node above the frontier: its box from two of
//                  those unions and the whole-block boxes between them; in a
//                  build also the nodes' places in the sibling-pair copy
//   copies         the traversal copies of the node array, four-child records
//                  (wide.hpp) and sibling pairs, each before the first query that
//                  reads it (tree_copies)
// Refit runs only local (bounds phase) + top_boxes.
//
// No box crosses workgroups through a counter: every hand-off between
// workgroups is a kernel boundary, so no agent-scope release/acquire (an L2
// write-back + invalidate on this chip) is issued per node. Every union keeps
// its operands in leaf order (box_join is the host's order-sensitive fminf /
// fmaxf), so each box has the bits of the host's recursive union.
//
// Algorithms follow the reference: Morton quantisation
// src/bvh/cpu_lbvh_builder.h:37-61 (device twin src/bvh/gpu_bvh.cu:135-149),
// stable key order src/bvh/cpu_lbvh_builder.h:212-216, Karras 2012 range/split
// with merged keys :63-131, internal box = union of children :139-159
// (union_aabb(left, right), src/core/aabb.cuh:113-115).
#include "lux_runtime.hpp"
#include "wide.hpp"

namespace lux {
namespace {

constexpr int kBlock = 256;
constexpr int kSortItems = 8;
constexpr int kSortTile = kBlock * kSortItems;  // 2048 keys per tile
constexpr int kRadix = 256;
constexpr int kPasses = 4;                      // 4 x 8 bits cover the 30-bit codes
constexpr int kReduceBlocksMax = 1024;
constexpr uint32_t kSpinLimit = 1u << 22;

// ---------------------------------------------------------------------------
// block-wide helpers (256 threads = 4 waves of 64)
// ---------------------------------------------------------------------------
__device__ __forceinline__ uint32_t wave_incl_scan(uint32_t x) {
    uint32_t lane = lane_id();
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
        uint32_t y = __shfl_up(x, off, 64);
        if (lane >= uint32_t(off)) x += y;
    }
    return x;
}

// Exclusive scan of one value per thread over a 256-thread block.
__device__ __forceinline__ uint32_t block_excl_scan(uint32_t x, uint32_t* s_tmp /*4 words*/) {
    uint32_t incl = wave_incl_scan(x);
    uint32_t wave = threadIdx.x >> 6;
    if (lane_id() == 63) s_tmp[wave] = incl;
    __syncthreads();
    uint32_t add = 0;
    for (uint32_t w = 0; w < wave; ++w) add += s_tmp[w];
    __syncthreads();
    return incl - x + add;
}

struct BoxIds {
    float lx, ly, lz, hx, hy, hz;
    int32_t imin, imax;
};

__device__ __forceinline__ void fold(BoxIds& a, const BoxIds& b) {
    a.lx = fminf(a.lx, b.lx);
    a.ly = fminf(a.ly, b.ly);
    a.lz = fminf(a.lz, b.lz);
    a.hx = fmaxf(a.hx, b.hx);
    a.hy = fmaxf(a.hy, b.hy);
    a.hz = fmaxf(a.hz, b.hz);
    a.imin = min(a.imin, b.imin);
    a.imax = max(a.imax, b.imax);
}

__device__ __forceinline__ BoxIds boxids_empty() {
    return BoxIds{INFINITY, INFINITY, INFINITY, -INFINITY, -INFINITY, -INFINITY, INT32_MAX, INT32_MIN};
}

// Block-wide fold of one BoxIds per thread; result valid in thread 0.
__device__ __forceinline__ BoxIds block_fold(BoxIds v) {
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
        BoxIds o;
        o.lx = __shfl_xor(v.lx, off, 64);
        o.ly = __shfl_xor(v.ly, off, 64);
        o.lz = __shfl_xor(v.lz, off, 64);
        o.hx = __shfl_xor(v.hx, off, 64);
        o.hy = __shfl_xor(v.hy, off, 64);
        o.hz = __shfl_xor(v.hz, off, 64);
        o.imin = __shfl_xor(v.imin, off, 64);
        o.imax = __shfl_xor(v.imax, off, 64);
        fold(v, o);
    }
    __shared__ BoxIds s_w[kBlock / 64];
    if (lane_id() == 0) s_w[threadIdx.x >> 6] = v;
    __syncthreads();
    if (threadIdx.x == 0)
        for (int w = 1; w < kBlock / 64; ++w) fold(v, s_w[w]);
    __syncthreads();
    return v;
}

// ---------------------------------------------------------------------------
// 1. root bounds partials (+ optional copy of the input into the handle)
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(kBlock) void k_root_partials(const lux_aabb* __restrict__ in_boxes,
                                                          const int32_t* __restrict__ in_ids,
                                                          lux_aabb* __restrict__ boxes,
                                                          int32_t* __restrict__ ids, int copy, int n,
                                                          BoxIds* __restrict__ partials,
                                                          uint32_t* __restrict__ hist,
                                                          DevInfo* __restrict__ info) {
    BoxIds acc = boxids_empty();
    for (int i = blockIdx.x * kBlock + threadIdx.x; i < n; i += gridDim.x * kBlock) {
        lux_aabb b = in_boxes[i];
        int32_t id = in_ids[i];
        if (copy) {
            boxes[i] = b;
            ids[i] = id;
        }
        BoxIds v{b.p_min.x, b.p_min.y, b.p_min.z, b.p_max.x, b.p_max.y, b.p_max.z, id, id};
        fold(acc, v);
    }
    acc = block_fold(acc);
    if (threadIdx.x == 0) partials[blockIdx.x] = acc;
    if (blockIdx.x == 0) {
        for (int w = threadIdx.x; w < kPasses * kRadix; w += kBlock) hist[w] = 0;
        if (threadIdx.x == 0) {
            info->max_depth = 0;
        }
    }
}

// ---------------------------------------------------------------------------
// 2. Morton codes + digit histograms
// ---------------------------------------------------------------------------
// Spread the 10 low bits of v to every third bit (bit k -> bit 3k).
__device__ __forceinline__ uint32_t spread_bits3(uint32_t v) {
    v &= 0x3ffu;
    v = (v | (v << 16)) & 0x030000ffu;
    v = (v | (v << 8)) & 0x0300f00fu;
    v = (v | (v << 4)) & 0x030c30c3u;
    v = (v | (v << 2)) & 0x09249249u;
    return v;
}

__device__ __forceinline__ uint32_t quantize10(float value) {
    value = fmaxf(0.0f, fminf(1023.0f, value * 1024.0f));
    return uint32_t(value);
}

__device__ __forceinline__ uint32_t morton30(const lux_aabb& root, const lux_aabb& b) {
    // centroid = (p_min + p_max) * 0.5, normalized_offset against the root box
    float cx = (b.p_min.x + b.p_max.x) * 0.5f;
    float cy = (b.p_min.y + b.p_max.y) * 0.5f;
    float cz = (b.p_min.z + b.p_max.z) * 0.5f;
    float dx = root.p_max.x - root.p_min.x;
    float dy = root.p_max.y - root.p_min.y;
    float dz = root.p_max.z - root.p_min.z;
    float ox = dx > 0 ? (cx - root.p_min.x) / dx : 0.5f;
    float oy = dy > 0 ? (cy - root.p_min.y) / dy : 0.5f;
    float oz = dz > 0 ? (cz - root.p_min.z) / dz : 0.5f;
    return (spread_bits3(quantize10(ox)) << 2) | (spread_bits3(quantize10(oy)) << 1) |
           spread_bits3(quantize10(oz));
}

__global__ __launch_bounds__(kBlock) void k_morton_hist(const lux_aabb* __restrict__ boxes, int n,
                                                        const BoxIds* __restrict__ partials,
                                                        int num_partials, DevInfo* __restrict__ info,
                                                        uint32_t* __restrict__ keys,
                                                        uint32_t* __restrict__ vals,
                                                        uint32_t* hist) {
    __shared__ uint32_t s_hist[kPasses * kRadix];
    __shared__ lux_aabb s_root;
    for (int w = threadIdx.x; w < kPasses * kRadix; w += kBlock) s_hist[w] = 0;
    // Every block folds the (at most 1024) partials itself: exact min/max, so all
    // blocks get the same root box without a cross-block hand-off.
    BoxIds acc = boxids_empty();
    for (int i = threadIdx.x; i < num_partials; i += kBlock) fold(acc, partials[i]);
    acc = block_fold(acc);
    if (threadIdx.x == 0) {
        lux_aabb r;
        r.p_min = lux_vec3{acc.lx, acc.ly, acc.lz};
        r.p_max = lux_vec3{acc.hx, acc.hy, acc.hz};
        s_root = r;
        if (blockIdx.x == 0) {
            info->root = r;
            info->id_min = acc.imin;
            info->id_max = acc.imax;
            if (acc.imin < 0) info->error |= kErrNegativeId;
        }
    }
    __syncthreads();
    const lux_aabb root = s_root;
    for (int i = blockIdx.x * kBlock + threadIdx.x; i < n; i += gridDim.x * kBlock) {
        uint32_t c = morton30(root, boxes[i]);
        keys[i] = c;
        vals[i] = uint32_t(i);
#pragma unroll
        for (int p = 0; p < kPasses; ++p) atomicAdd(&s_hist[p * kRadix + ((c >> (8 * p)) & 0xffu)], 1u);
    }
    __syncthreads();
    for (int w = threadIdx.x; w < kPasses * kRadix; w += kBlock) {
        uint32_t c = s_hist[w];
        if (c) __hip_atomic_fetch_add(&hist[w], c, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
}

// Ray-order keys: the direction octant (sign bits of d) in bits 27..29 above
// the top 27 bits of the 30-bit Morton code of the ray origin in the tree's
// root box (origins outside clamp to the boundary cells), payload = ray index,
// and the histograms of the digits at bits 14..21 and 22..29 (hist zeroed
// before). Sorting on bits 14..29 groups rays by octant, then by origin cell
// (13 Morton bits). On 2^22 random rays over 2^20 triangles this measured
// 5.12 ms closest hit and 5.11 ms any hit against 5.37 / 5.43 ms in origin-only
// order; 2 bits of quantised direction per axis instead of the octant measured
// slower (5.42 / 5.75 ms).
__global__ __launch_bounds__(kBlock) void k_ray_keys(const lux_ray* __restrict__ rays, int n,
                                                     const DevInfo* __restrict__ info,
                                                     uint32_t* __restrict__ keys, uint32_t* __restrict__ vals,
                                                     uint32_t* hist) {
    __shared__ uint32_t s_hist[2 * kRadix];
    for (int w = threadIdx.x; w < 2 * kRadix; w += kBlock) s_hist[w] = 0;
    __syncthreads();
    const lux_aabb root = info->root;
    const float dx = root.p_max.x - root.p_min.x, dy = root.p_max.y - root.p_min.y,
                dz = root.p_max.z - root.p_min.z;
    for (int i = blockIdx.x * kBlock + threadIdx.x; i < n; i += gridDim.x * kBlock) {
        const lux_vec3 o = rays[i].origin;
        float ox = dx > 0 ? (o.x - root.p_min.x) / dx : 0.5f;
        float oy = dy > 0 ? (o.y - root.p_min.y) / dy : 0.5f;
        float oz = dz > 0 ? (o.z - root.p_min.z) / dz : 0.5f;
        // NaN origins quantize to cell 0 (fmaxf drops the NaN)
        uint32_t c = (spread_bits3(quantize10(ox)) << 2) | (spread_bits3(quantize10(oy)) << 1) |
                     spread_bits3(quantize10(oz));
        const lux_vec3 d = rays[i].direction;
        const uint32_t octant = (d.x < 0 ? 4u : 0u) | (d.y < 0 ? 2u : 0u) | (d.z < 0 ? 1u : 0u);
        c = (octant << 27) | (c >> 3);
        keys[i] = c;
        vals[i] = uint32_t(i);
        atomicAdd(&s_hist[(c >> 14) & 0xffu], 1u);
        atomicAdd(&s_hist[kRadix + ((c >> 22) & 0xffu)], 1u);
    }
    __syncthreads();
    for (int w = threadIdx.x; w < 2 * kRadix; w += kBlock) {
        uint32_t c = s_hist[w];
        if (c) __hip_atomic_fetch_add(&hist[w], c, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
}

__global__ void k_zero_u32(uint32_t* p, int n) {
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) p[i] = 0;
}

// What the kernels of a new tree expect to be zero: look-back words (epoch 0 is
// never used), tile tickets, the pair counter and the tree's info. A kernel on
// the stream that builds the tree: hipMemset is ordered on the null stream,
// which no stream of the library waits for, and returns before it is done
// (16 bytes: 5 us; the fill itself came 2.6 ms later on a chip kept busy by another
// stream). A pass that starts on another tree's tickets takes a tile out of range.
__global__ void k_clear_tree(uint64_t* __restrict__ status, int words, uint32_t* __restrict__ tickets,
                             int32_t* __restrict__ counter, DevInfo* __restrict__ info) {
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < words; i += gridDim.x * blockDim.x) status[i] = 0;
    if (blockIdx.x == 0) {
        if (threadIdx.x < 4) {
            tickets[threadIdx.x] = 0;
            counter[threadIdx.x] = 0;
        }
        if (threadIdx.x < sizeof(DevInfo) / 4) reinterpret_cast<uint32_t*>(info)[threadIdx.x] = 0;
    }
}

// ---------------------------------------------------------------------------
// 3. one stable LSD radix pass (8-bit digit) with decoupled look-back
// ---------------------------------------------------------------------------
// Look-back word: [epoch:32][flag:2][count:30]. flag 1 = tile aggregate only,
// flag 2 = inclusive prefix over tiles 0..t. Words from an older pass carry an
// older epoch and read as "not ready", so the array is never cleared.
constexpr uint64_t kFlagAggregate = 1;
constexpr uint64_t kFlagInclusive = 2;
// Predecessors read at once by a tile's look-back. One pass over 2^20 keys (512
// tiles) took 27.5 / 24.7 / 25.0 / 27.2 us with 1 / 4 / 8 / 16, over 2^22 rays
// 68 / 64 / 64 / 69 us.
constexpr int kLookback = 4;

__device__ __forceinline__ uint64_t pack_status(uint32_t epoch, uint64_t flag, uint32_t count) {
    return (uint64_t(epoch) << 32) | (flag << 30) | uint64_t(count & 0x3fffffffu);
}

__global__ __launch_bounds__(kBlock) void k_sort_pass(const uint32_t* __restrict__ keys_in,
                                                      const uint32_t* __restrict__ vals_in,
                                                      uint32_t* __restrict__ keys_out,
                                                      uint32_t* __restrict__ vals_out, int n,
                                                      int shift, const uint32_t* __restrict__ hist,
                                                      uint64_t* status, uint32_t* ticket,
                                                      uint32_t epoch, int num_tiles,
                                                      DevInfo* info) {
    __shared__ uint32_t s_wave_cnt[4][kRadix];
    __shared__ uint32_t s_tile_start[kRadix];
    __shared__ uint32_t s_base[kRadix];
    __shared__ uint32_t s_keys[kSortTile];
    __shared__ uint32_t s_vals[kSortTile];
    __shared__ uint32_t s_tmp[4];
    __shared__ uint32_t s_ticket;

    const uint32_t tid = threadIdx.x;
    const uint32_t wave = tid >> 6;
    const uint32_t lane = lane_id();

    if (tid == 0) s_ticket = __hip_atomic_fetch_add(ticket, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    for (int w = tid; w < 4 * kRadix; w += kBlock) (&s_wave_cnt[0][0])[w] = 0;
    __syncthreads();
    const uint32_t tile = s_ticket;
    if (tile >= uint32_t(num_tiles)) {  // a ticket counter that did not start at zero
        if (tid == 0) set_error(info, kErrSpinLimit);
        return;
    }
    // Tickets are handed out in start order, so a tile only ever waits on tiles
    // that are already running. The last ticket resets the counter for the next
    // launch on this stream.
    if (tid == 0 && tile == uint32_t(num_tiles - 1))
        __hip_atomic_store(ticket, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);

    const int tile_base = int(tile) * kSortTile;
    uint32_t k[kSortItems], v[kSortItems], rank[kSortItems];
#pragma unroll
    for (int r = 0; r < kSortItems; ++r) {
        int g = tile_base + int(wave) * (64 * kSortItems) + r * 64 + int(lane);
        bool valid = g < n;
        k[r] = valid ? keys_in[g] : 0u;
        v[r] = valid ? vals_in[g] : 0u;
    }
    // Rank each key among equal digits: earlier rounds of this wave via the
    // running per-wave counter, earlier lanes of this round via ballot matching.
    volatile uint32_t* wave_cnt = &s_wave_cnt[wave][0];
#pragma unroll
    for (int r = 0; r < kSortItems; ++r) {
        int g = tile_base + int(wave) * (64 * kSortItems) + r * 64 + int(lane);
        bool valid = g < n;
        uint32_t dig = (k[r] >> shift) & 0xffu;
        uint64_t peers = ballot64(valid);
#pragma unroll
        for (int b = 0; b < 8; ++b) {
            bool bit = (dig >> b) & 1u;
            uint64_t m = ballot64(bit);
            peers &= bit ? m : ~m;
        }
        uint32_t prior = valid ? wave_cnt[dig] : 0u;
        rank[r] = prior + uint32_t(__popcll(peers & lanemask_lt()));
        bool last_of_group = valid && ((peers >> lane) == 1ull);
        __builtin_amdgcn_wave_barrier();
        if (last_of_group) wave_cnt[dig] = prior + uint32_t(__popcll(peers));
        __builtin_amdgcn_wave_barrier();
    }
    __syncthreads();

    // Per digit (thread = digit): wave offsets and the tile total.
    const uint32_t dgt = tid;
    uint32_t c0 = s_wave_cnt[0][dgt], c1 = s_wave_cnt[1][dgt], c2 = s_wave_cnt[2][dgt],
             c3 = s_wave_cnt[3][dgt];
    uint32_t total = c0 + c1 + c2 + c3;
    uint64_t* my_status = status + size_t(tile) * kRadix + dgt;
    __hip_atomic_store(my_status, pack_status(epoch, tile == 0 ? kFlagInclusive : kFlagAggregate, total),
                       __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    s_wave_cnt[0][dgt] = 0;
    s_wave_cnt[1][dgt] = c0;
    s_wave_cnt[2][dgt] = c0 + c1;
    s_wave_cnt[3][dgt] = c0 + c1 + c2;

    uint32_t tile_start = block_excl_scan(total, s_tmp);
    uint32_t global_start = block_excl_scan(hist[dgt], s_tmp);

    uint32_t excl = 0;
    if (tile > 0) {
        int j = int(tile) - 1;
        uint32_t spins = 0;
        bool found = false;
        while (!found && j >= 0) {
            // the words of the next kLookback tiles at once: a word is an
            // uncached load past the XCD's L2, so one at a time the walk is a
            // chain of memory latencies
            uint64_t word[kLookback];
#pragma unroll
            for (int k = 0; k < kLookback; ++k) {
                const int jj = max(j - k, 0);
                word[k] = __hip_atomic_load(status + size_t(jj) * kRadix + dgt, __ATOMIC_RELAXED,
                                            __HIP_MEMORY_SCOPE_AGENT);
            }
            int used = 0;
#pragma unroll
            for (int k = 0; k < kLookback; ++k) {
                const uint64_t flag = (word[k] >> 30) & 3u;
                if (found || used < k || j - k < 0 || uint32_t(word[k] >> 32) != epoch || flag == 0) continue;
                excl += uint32_t(word[k] & 0x3fffffffu);
                found = flag == kFlagInclusive;
                used = k + 1;
            }
            j -= used;
            if (used == 0 && !found && j >= 0) {
                if (++spins > kSpinLimit) {
                    set_error(info, kErrSpinLimit);
                    break;
                }
                __builtin_amdgcn_s_sleep(1);
            }
        }
        __hip_atomic_store(my_status, pack_status(epoch, kFlagInclusive, excl + total),
                           __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    s_tile_start[dgt] = tile_start;
    s_base[dgt] = global_start + excl;
    __syncthreads();

    // Local scatter into LDS in digit order, then coalesced runs to HBM.
#pragma unroll
    for (int r = 0; r < kSortItems; ++r) {
        int g = tile_base + int(wave) * (64 * kSortItems) + r * 64 + int(lane);
        if (g < n) {
            uint32_t dig = (k[r] >> shift) & 0xffu;
            uint32_t pos = s_tile_start[dig] + s_wave_cnt[wave][dig] + rank[r];
            s_keys[pos] = k[r];
            s_vals[pos] = v[r];
        }
    }
    __syncthreads();
    int tile_count = min(kSortTile, n - tile_base);
    for (int i = tid; i < tile_count; i += kBlock) {
        uint32_t key = s_keys[i];
        uint32_t dig = (key >> shift) & 0xffu;
        uint32_t out = s_base[dig] + (uint32_t(i) - s_tile_start[dig]);
        if (out >= uint32_t(n)) {  // only after a failed look-back
            set_error(info, kErrSpinLimit);
            continue;
        }
        keys_out[out] = key;
        vals_out[out] = s_vals[i];
    }
}

// ---------------------------------------------------------------------------
// 4. Karras radix tree (+ frontier list)
// ---------------------------------------------------------------------------
// Leaves are grouped into blocks of kLocalLeaves consecutive sorted leaves. A
// node is LOCAL when its leaf range lies inside one block; a local node whose
// parent is not local is a FRONTIER node. Every internal node is either local
// (handled entirely by the workgroup of its block) or above the frontier (its
// range [first, last] has first / kLocalLeaves != last / kLocalLeaves).
constexpr int kLocalLeaves = 1024;

__device__ __forceinline__ int prefix_len(const uint32_t* __restrict__ codes, int a, int b) {
    uint64_t ka = (uint64_t(codes[a]) << 32) | uint64_t(uint32_t(a));
    uint64_t kb = (uint64_t(codes[b]) << 32) | uint64_t(uint32_t(b));
    return __clzll(ka ^ kb);  // a != b, so the keys differ
}

__global__ __launch_bounds__(kBlock) void k_karras(const uint32_t* __restrict__ codes, int n,
                                                   uint32_t* __restrict__ left,
                                                   uint32_t* __restrict__ right, uint32_t* parent,
                                                   uint32_t* leaf_parent,
                                                   uint32_t* __restrict__ first_out,
                                                   uint32_t* __restrict__ last_out) {
    int i = blockIdx.x * kBlock + threadIdx.x;
    if (i >= n - 1) return;
    int first, last;
    if (i == 0) {
        first = 0;
        last = n - 1;
        parent[0] = 0;
    } else {
        int dl = prefix_len(codes, i, i - 1);
        int dr = prefix_len(codes, i, i + 1);
        int dir = dr > dl ? 1 : -1;
        int dmin = min(dl, dr);
        int lmax = 2;
        for (;;) {
            int j = i + dir * lmax;
            if (j < 0 || j >= n || prefix_len(codes, i, j) <= dmin) break;
            lmax <<= 1;
        }
        int len = 0;
        for (int step = lmax >> 1; step > 0; step >>= 1) {
            int j = i + (len + step) * dir;
            if (j < 0 || j >= n) continue;
            if (prefix_len(codes, i, j) > dmin) len += step;
        }
        int other = i + len * dir;
        first = dir < 0 ? other : i;
        last = dir < 0 ? i : other;
    }
    int dnode = prefix_len(codes, first, last);
    int split = first, stride = last - first;
    do {
        stride = (stride + 1) >> 1;
        int mid = split + stride;
        if (mid < last && prefix_len(codes, first, mid) > dnode) split = mid;
    } while (stride > 1);

    uint32_t lchild, rchild;
    if (first == split) {
        lchild = kLeafBit | uint32_t(split);
        leaf_parent[split] = uint32_t(i);
    } else {
        lchild = uint32_t(split);
        parent[split] = uint32_t(i);
    }
    if (last == split + 1) {
        rchild = kLeafBit | uint32_t(split + 1);
        leaf_parent[split + 1] = uint32_t(i) | kLeafBit;
    } else {
        rchild = uint32_t(split + 1);
        parent[split + 1] = uint32_t(i) | kLeafBit;
    }
    left[i] = lchild;
    right[i] = rchild;
    first_out[i] = uint32_t(first);
    last_out[i] = uint32_t(last);
}

// ---------------------------------------------------------------------------
// 5. right-first preorder layout
// ---------------------------------------------------------------------------
// In right-first preorder a node X is preceded by its ancestors and by the right
// subtrees of the ancestors whose LEFT subtree holds X; those subtrees hold the
// n-1-last(X) leaves right of X. Hence
//     pre(X) = 2 (n - 1 - last(X)) + R(X),
// R(X) = number of ancestors whose right subtree holds X (right steps on the
// path to the root). Descending a right child adds one, so the nodes on the
// "right chain" above X (reached from X by right steps only) sit at pre(X) - 1,
// pre(X) - 2, ... Every internal node is on the right chain of exactly one leaf
// (its last leaf) and -- if it is above the frontier -- of exactly one frontier
// node. Subtree size = 2 (last - first + 1) - 1 and escape = pre + size.
//
// top_layout: one thread per internal node above the frontier walks to the
// root counting right steps R and levels, stores pre(X) = 2 (n - 1 - last) + R,
// and hands each local child F (a frontier node) R(F) = R(X) + [F is X's right
// child] | (depth(X) + 1) << 16, which the local pass adds to the steps inside
// the block.
__global__ __launch_bounds__(kBlock) void k_top_layout(int n, const uint32_t* __restrict__ parent,
                                                       const uint32_t* __restrict__ left,
                                                       const uint32_t* __restrict__ right,
                                                       const uint32_t* __restrict__ first_of,
                                                       const uint32_t* __restrict__ last_of,
                                                       uint32_t* __restrict__ rtop_int,
                                                       uint32_t* __restrict__ rtop_leaf,
                                                       int32_t* __restrict__ pre_internal, DevInfo* info) {
    const int total = 2 * n - 1;
    for (int i = blockIdx.x * kBlock + threadIdx.x; i < n - 1; i += gridDim.x * kBlock) {
        const uint32_t first = first_of[i], last = last_of[i];
        if (first / kLocalLeaves == last / kLocalLeaves) continue;
        uint32_t rights = 0, depth = 0, p = uint32_t(i);
        bool bad = false;
        while (p != 0) {
            if (depth > 64u) {  // a merged-key tree is at most 64 internal nodes deep
                bad = true;
                break;
            }
            const uint32_t pp = parent[p];
            rights += pp >> 31;
            p = pp & kIndexMask;
            ++depth;
            if (p >= uint32_t(n - 1)) {
                bad = true;
                break;
            }
        }
        const int pos = 2 * (n - 1 - int(last)) + int(rights);
        if (bad || pos < 0 || pos >= total) {
            set_error(info, kErrClimbLimit);
            continue;
        }
        pre_internal[i] = pos;
        const uint32_t kids[2] = {left[i], right[i]};
        for (uint32_t side = 0; side < 2; ++side) {
            const uint32_t c = kids[side];
            const uint32_t idx = c & kIndexMask;
            const bool leaf = c & kLeafBit;
            const uint32_t cf = leaf ? idx : first_of[idx], cl = leaf ? idx : last_of[idx];
            if (cf / kLocalLeaves != cl / kLocalLeaves) continue;  // above the frontier too
            const uint32_t packed = (rights + side) | ((depth + 1) << 16);
            if (leaf)
                rtop_leaf[idx] = packed;
            else
                rtop_int[idx] = packed;
        }
    }
}

// ---------------------------------------------------------------------------
// 6. local pass: one workgroup per leaf block
// ---------------------------------------------------------------------------
// kMode 0: build (layout, then boxes from the handle's input copy)
// kMode 1: refit from boxes        kMode 2: refit from triangles
//
// The block's tree data sits in LDS (parent links of the internal nodes and
// leaves with index in [lo, hi] -- every local internal node has its index in
// its own range, so inside the block -- their leaf counts and preorder
// positions), so the climbs below touch global memory only for the leaf input
// and the one 32-byte write of each finished node.
//
// Bounds: every local internal node gets exactly two arrivals from threads of
// this workgroup; each leaves its box in its side's LDS slot and bumps the
// node's 8-bit arrival counter. The arrival that reads 0 stops; the other
// unions left-then-right, writes the node and climbs on. A climb stops at a
// frontier node (its parent lies above the block); the frontier nodes are then
// put in leaf order and folded into
//   edge_boxes[2 first]     union from a left-child frontier node's first leaf
//                           to the end of the block
//   edge_boxes[2 last + 1]  union from the start of the block to a right-child
//                           frontier node's last leaf
//   block_boxes[block]      union of the whole block
// which is all top_boxes needs. A block holds at most 128 frontier nodes: each
// is a child of a node whose range crosses one of the block's two edges, and
// the nodes over an edge lie on one root path, at most 64 long (a child's
// common key prefix is longer than its parent's, and keys have 64 bits).
constexpr int kMaxFrontier = 128;

struct FrontierRec {
    lux_aabb box;
    uint32_t span;  // first leaf - lo | (last leaf - lo) << 10 | is_left_child << 20
};

__device__ __forceinline__ void store_node(lux_bvh_node* nodes, int pos, const lux_aabb& b, int32_t prim,
                                           int size, int total) {
    const int esc = pos + size;
    float4* p = reinterpret_cast<float4*>(nodes + pos);
    p[0] = make_float4(b.p_min.x, b.p_min.y, b.p_min.z, b.p_max.x);
    p[1] = make_float4(b.p_max.y, b.p_max.z, __int_as_float(prim), __int_as_float(esc < total ? esc : -1));
}

// kLocalThreads: see launch_local.
template <int kMode, int kLocalThreads>
__global__ __launch_bounds__(kLocalThreads) void k_local(
    int n, const uint32_t* __restrict__ sorted_input, const int32_t* __restrict__ ids,
    const lux_aabb* __restrict__ src_boxes, const lux_triangle* __restrict__ src_tris,
    lux_aabb* own_boxes, int write_back, const uint32_t* __restrict__ parent,
    const uint32_t* __restrict__ leaf_parent, const uint32_t* __restrict__ first_of,
    const uint32_t* __restrict__ last_of, const uint32_t* __restrict__ rtop_int,
    const uint32_t* __restrict__ rtop_leaf, lux_bvh_node* __restrict__ nodes, int32_t* __restrict__ pre_internal,
    int32_t* __restrict__ pre_leaf, lux_aabb* __restrict__ edge_boxes, lux_aabb* __restrict__ block_boxes,
    DevInfo* info) {
    __shared__ lux_aabb s_slot[kLocalLeaves][2];
    __shared__ uint32_t s_arrive[kLocalLeaves / 4];
    __shared__ uint32_t s_par[kLocalLeaves];
    __shared__ uint32_t s_lpar[kLocalLeaves];
    __shared__ uint16_t s_leaves[kLocalLeaves];  // leaf count of a local internal node, 0 if not local
    __shared__ int32_t s_pre_int[kLocalLeaves];
    __shared__ int32_t s_pre_leaf[kLocalLeaves];
    __shared__ FrontierRec s_fr[kMaxFrontier];
    __shared__ uint8_t s_order[kMaxFrontier];
    __shared__ uint32_t s_fcount;
    const int lo = blockIdx.x * kLocalLeaves;
    const int hi = min(lo + kLocalLeaves, n) - 1;
    const int cnt = hi - lo + 1;
    const int total = 2 * n - 1;
    const int tid = threadIdx.x;

    for (int k = tid; k < kLocalLeaves / 4; k += kLocalThreads) s_arrive[k] = 0;
    if (tid < kMaxFrontier) s_order[tid] = 0;
    if (tid == 0) s_fcount = 0;
    for (int k = tid; k < cnt; k += kLocalThreads) {
        const int i = lo + k;
        s_lpar[k] = leaf_parent[i];
        uint32_t leaves = 0, par = 0;
        if (i <= n - 2) {
            const uint32_t f = first_of[i], l = last_of[i];
            if (int(f) >= lo && int(l) <= hi) leaves = l - f + 1;
            par = parent[i];
        }
        s_leaves[k] = uint16_t(leaves);
        s_par[k] = par;
        if (kMode != 0) {
            s_pre_leaf[k] = pre_leaf[i];
            s_pre_int[k] = leaves ? pre_internal[i] : -1;
        }
    }
    __syncthreads();
    auto local_leaves = [&](uint32_t p) -> uint32_t {
        const uint32_t r = p - uint32_t(lo);
        return r < uint32_t(cnt) ? uint32_t(s_leaves[r]) : 0u;
    };

    if (kMode == 0) {
        uint32_t max_depth = 0;
        for (int k = tid; k < cnt; k += kLocalThreads) {
            const int j = lo + k;
            const uint32_t lp = s_lpar[k];
            uint32_t side = lp >> 31;
            uint32_t p = lp & kIndexMask;
            int rights = 0, chain = 0;
            uint32_t all_right = 1, steps = 0;
            bool reached_root = false, f_is_leaf = true, bad = false;
            uint32_t f = uint32_t(j);
            for (int guard = 0;; ++guard) {
                if (!local_leaves(p)) break;
                if (guard > kLocalLeaves) {
                    bad = true;
                    break;
                }
                rights += int(side);
                all_right &= side;
                chain += int(all_right);
                ++steps;
                f_is_leaf = false;
                f = p;
                if (p == 0) {
                    reached_root = true;
                    break;
                }
                const uint32_t pp = s_par[p - uint32_t(lo)];
                side = pp >> 31;
                p = pp & kIndexMask;
            }
            const uint32_t top = reached_root ? 0u : (f_is_leaf ? rtop_leaf[f] : rtop_int[f]);
            int pos = 2 * (n - 1 - j) + rights + int(top & 0xffffu);
            max_depth = max(max_depth, steps + (top >> 16));
            if (bad || pos - chain < 0 || pos >= total) {  // no early return: a barrier follows
                set_error(info, kErrClimbLimit);
                s_pre_leaf[k] = -1;
                continue;
            }
            s_pre_leaf[k] = pos;
            pre_leaf[j] = pos;
            uint32_t c_node = lp & kIndexMask;
            for (int c = 0; c < chain; ++c) {
                --pos;
                s_pre_int[c_node - uint32_t(lo)] = pos;
                pre_internal[c_node] = pos;
                if (c + 1 < chain) c_node = s_par[c_node - uint32_t(lo)] & kIndexMask;
            }
        }
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) max_depth = max(max_depth, uint32_t(__shfl_xor(int(max_depth), off, 64)));
        if (lane_id() == 0)
            __hip_atomic_fetch_max(&info->max_depth, max_depth, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __syncthreads();  // every preorder position of the block is in LDS
    }

    for (int k = tid; k < cnt; k += kLocalThreads) {
        const int j = lo + k;
        const uint32_t in = sorted_input[j];
        if (in >= uint32_t(n)) {  // only after a failed sort
            set_error(info, kErrSpinLimit);
            continue;
        }
        lux_aabb box = kMode == 2 ? tri_box(src_tris[in]) : src_boxes[in];
        if (write_back) own_boxes[in] = box;
        int pre = s_pre_leaf[k];
        if (uint32_t(pre) >= uint32_t(total)) {
            set_error(info, kErrClimbLimit);
            continue;
        }
        store_node(nodes, pre, box, ids[in], 1, total);
        uint32_t lp = s_lpar[k];
        uint32_t first_rel = uint32_t(k), last_rel = uint32_t(k);
        for (int guard = 0;; ++guard) {
            const uint32_t side = lp >> 31;
            const uint32_t p = lp & kIndexMask;
            const uint32_t leaves = local_leaves(p);
            if (!leaves) {  // frontier node: its parent lies above the block
                const uint32_t e = __hip_atomic_fetch_add(&s_fcount, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
                if (e < uint32_t(kMaxFrontier)) {
                    s_fr[e].box = box;
                    s_fr[e].span = first_rel | (last_rel << 10) | ((side ^ 1u) << 20);
                } else {
                    set_error(info, kErrClimbLimit);
                }
                break;
            }
            if (guard > kLocalLeaves) {
                set_error(info, kErrClimbLimit);
                break;
            }
            const uint32_t slot = p - uint32_t(lo);
            s_slot[slot][side] = box;
            // The hand-off is LDS only: order the slot write before the counter
            // and the counter before the sibling's slot read, without waiting
            // for this thread's node stores to reach memory.
            const uint32_t sh = 8u * (slot & 3u);
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
            const uint32_t old = __hip_atomic_fetch_add(&s_arrive[slot >> 2], 1u << sh, __ATOMIC_RELAXED,
                                                        __HIP_MEMORY_SCOPE_WORKGROUP);
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
            if (((old >> sh) & 0xffu) == 0) break;
            box = side ? box_join(s_slot[slot][0], box) : box_join(box, s_slot[slot][1]);
            if (side)
                first_rel = last_rel + 1 - leaves;
            else
                last_rel = first_rel + leaves - 1;
            pre = s_pre_int[slot];
            if (uint32_t(pre) >= uint32_t(total)) {
                set_error(info, kErrClimbLimit);
                break;
            }
            store_node(nodes, pre, box, -1, int(2 * leaves - 1), total);
            if (p == 0) {
                info->root = box;
                break;
            }
            lp = s_par[slot];
        }
    }
    __syncthreads();  // every frontier record is in LDS

    const uint32_t fc = min(s_fcount, uint32_t(kMaxFrontier));
    for (uint32_t e = tid; e < fc; e += kLocalThreads) {
        const uint32_t fe = s_fr[e].span & 1023u;
        uint32_t rank = 0;
        for (uint32_t o = 0; o < fc; ++o) rank += (s_fr[o].span & 1023u) < fe ? 1u : 0u;
        s_order[rank] = uint8_t(e);
    }
    __syncthreads();
    if (tid == 0) {  // prefix unions, left to right
        lux_aabb acc = box_empty();
        for (uint32_t r = 0; r < fc; ++r) {
            const FrontierRec& f = s_fr[s_order[r]];
            acc = r ? box_join(acc, f.box) : f.box;
            const int at = lo + int((f.span >> 10) & 1023u);
            if (!(f.span >> 20) && at < n) edge_boxes[2 * size_t(at) + 1] = acc;
        }
        if (fc) block_boxes[blockIdx.x] = acc;
    } else if (tid == 64) {  // suffix unions, right to left (second wave)
        lux_aabb acc = box_empty();
        for (uint32_t r = fc; r-- > 0;) {
            const FrontierRec& f = s_fr[s_order[r]];
            acc = r + 1 < fc ? box_join(f.box, acc) : f.box;
            const int at = lo + int(f.span & 1023u);
            if ((f.span >> 20) && at < n) edge_boxes[2 * size_t(at)] = acc;
        }
    }
}

// Slots of the children of the internal node at preorder position k, whose leaf
// range ends at `last` and whose left child's ends at `split`. In right-first
// preorder the nodes before it are the n-1-last leaves right of its range and
// k-(n-1-last) internal nodes, which is its internal rank r. Its children go to
// the pair r+1: the right child (position k+1, 2 (last - split) - 1 nodes) at slot
// 2r+2, the left child (behind it) at slot 2r+3.
__device__ __forceinline__ void pair_slots(int n, int k, uint32_t split, uint32_t last,
                                           uint32_t* __restrict__ pair_pos, DevInfo* info) {
    const int node_count = 2 * n - 1;
    const int rank = k - (n - 1 - int(last));
    const int left = k + 2 * int(last - split);
    if (k < 0 || rank < 0 || rank >= n - 1 || left <= k + 1 || left >= node_count) {
        set_error(info, kErrWalkOrder);
        return;
    }
    pair_pos[k + 1] = uint32_t(2 * rank + 2);
    pair_pos[left] = uint32_t(2 * rank + 3);
}

// ---------------------------------------------------------------------------
// 7. top boxes: one wave per node above the frontier
// ---------------------------------------------------------------------------
// A node X above the frontier covers leaves [first, last] that start inside
// leaf block bf and end inside block bl > bf: its box is the union from
// `first` to the end of bf (the suffix stored at its leftmost frontier node, a
// left child), the whole blocks between, and the union from the start of bl to
// `last` (the prefix at its rightmost frontier node, a right child). The
// blocks between are folded in contiguous runs, lane by lane, then across the
// wave with lower lanes on the left, so the host's left-to-right order holds.
// kLayout (build): every lane also places its node's children in the
// sibling-pair copy; a launch of its own for that took 13 us at 2^20 leaves and
// 5 us at 100 000.
__device__ __forceinline__ lux_aabb shfl_down_box(const lux_aabb& b, int off) {
    lux_aabb r;
    r.p_min.x = __shfl_down(b.p_min.x, off, 64);
    r.p_min.y = __shfl_down(b.p_min.y, off, 64);
    r.p_min.z = __shfl_down(b.p_min.z, off, 64);
    r.p_max.x = __shfl_down(b.p_max.x, off, 64);
    r.p_max.y = __shfl_down(b.p_max.y, off, 64);
    r.p_max.z = __shfl_down(b.p_max.z, off, 64);
    return r;
}

template <bool kLayout>
__global__ __launch_bounds__(kBlock) void k_top_boxes(int n, const uint32_t* __restrict__ first_of,
                                                      const uint32_t* __restrict__ last_of,
                                                      const uint32_t* __restrict__ left,
                                                      uint32_t* __restrict__ pair_pos,
                                                      const int32_t* __restrict__ pre_internal,
                                                      const lux_aabb* __restrict__ edge_boxes,
                                                      const lux_aabb* __restrict__ block_boxes,
                                                      lux_bvh_node* __restrict__ nodes, DevInfo* info) {
    const uint32_t lane = lane_id();
    const int waves = gridDim.x * (kBlock / 64);
    const int total = 2 * n - 1;
    // each wave scans 64 internal nodes at a time and handles the ones above
    // the frontier (about one in a hundred) one after another, whole-wave
    for (int base = (blockIdx.x * (kBlock / 64) + int(threadIdx.x >> 6)) * 64; base < n - 1; base += waves * 64) {
        const int i = base + int(lane);
        uint32_t my_first = 0, my_last = 0;
        if (i < n - 1) {
            my_first = first_of[i];
            my_last = last_of[i];
            if (kLayout) {
                if (i == 0) pair_pos[0] = 0;  // the root stays at slot 0
                pair_slots(n, pre_internal[i], left[i] & kIndexMask, my_last, pair_pos, info);
            }
        }
        uint64_t todo = __ballot(i < n - 1 && my_first / kLocalLeaves != my_last / kLocalLeaves);
        while (todo) {
            const int l = __ffsll((unsigned long long)todo) - 1;
            todo &= todo - 1;
            const uint32_t x = uint32_t(base + l);
            const uint32_t first = uint32_t(__shfl(int(my_first), l, 64));
            const uint32_t last = uint32_t(__shfl(int(my_last), l, 64));
            const uint32_t bf = first / uint32_t(kLocalLeaves), bl = last / uint32_t(kLocalLeaves);
            const uint32_t m = bl - bf - 1;  // whole blocks between (bl > bf)
            const uint32_t per = (m + 63u) / 64u;
            const uint32_t b0 = bf + 1 + lane * per;
            const uint32_t b1 = min(b0 + per, bl);
            lux_aabb acc = box_empty();
            int have = 0;
            for (uint32_t b = b0; b < b1; ++b) {
                const lux_aabb bb = block_boxes[b];
                acc = have ? box_join(acc, bb) : bb;
                have = 1;
            }
#pragma unroll
            for (int off = 1; off < 64; off <<= 1) {
                const lux_aabb o = shfl_down_box(acc, off);
                const int o_have = __shfl_down(have, off, 64);
                if ((lane & uint32_t(2 * off - 1)) == 0 && lane + uint32_t(off) < 64u && o_have) {
                    acc = have ? box_join(acc, o) : o;
                    have = 1;
                }
            }
            if (lane == 0) {
                const int pre = pre_internal[x];
                if (uint32_t(pre) >= uint32_t(total)) {
                    set_error(info, kErrClimbLimit);
                } else {
                    lux_aabb box = edge_boxes[2 * size_t(first)];
                    if (have) box = box_join(box, acc);
                    box = box_join(box, edge_boxes[2 * size_t(last) + 1]);
                    store_node(nodes, pre, box, -1, int(2 * (last - first + 1) - 1), total);
                    if (x == 0) info->root = box;
                }
            }
        }
    }
}

__global__ void k_single_leaf(const lux_aabb* __restrict__ src_boxes,
                              const lux_triangle* __restrict__ src_tris, const int32_t* ids,
                              lux_aabb* own_boxes, int write_back, lux_bvh_node* nodes,
                              int32_t* pre_leaf, uint32_t* sorted_keys, uint32_t* sorted_input,
                              DevInfo* info, int layout) {
    lux_aabb b = src_tris ? tri_box(src_tris[0]) : src_boxes[0];
    if (write_back) own_boxes[0] = b;
    nodes[0].bounds = b;
    if (layout) {
        nodes[0].primitive_id = ids[0];
        nodes[0].escape = -1;
        pre_leaf[0] = 0;
        sorted_keys[0] = 0;
        sorted_input[0] = 0;
    }
    info->root = b;
}

template <typename T>
T* dalloc(size_t count) {
    void* p = nullptr;
    if (count == 0) count = 1;
    hipError_t e = hipMalloc(&p, count * sizeof(T));
    if (e != hipSuccess) throw Error(LUX_ERR_OUT_OF_MEMORY, std::string("hipMalloc failed: ") + hipGetErrorString(e));
    return static_cast<T*>(p);
}

int reduce_blocks(int n) { return max(1, min(kReduceBlocksMax, div_up(n, kBlock * 4))); }
int sort_tiles(int n) { return max(1, div_up(n, kSortTile)); }

}  // namespace

// ---------------------------------------------------------------------------
// sibling-pair traversal copy of the node array
// ---------------------------------------------------------------------------
namespace {
// Pair positions of a tree of one leaf block (larger ones: k_top_boxes).
__global__ __launch_bounds__(kBlock) void k_pair_layout(int n, const uint32_t* __restrict__ left,
                                                        const uint32_t* __restrict__ last,
                                                        const int32_t* __restrict__ pre_internal,
                                                        uint32_t* __restrict__ pair_pos, DevInfo* info) {
    const int i = blockIdx.x * kBlock + threadIdx.x;
    if (i == 0) pair_pos[0] = 0;  // the root (leaf or internal) stays at slot 0
    if (i < n - 1) pair_slots(n, pre_internal[i], left[i] & kIndexMask, last[i], pair_pos, info);
}

// Copies every node to its slot: boxes and leaf ids as they are, internal
// nodes point at their right child's slot, escapes are translated to slots.
// Slot 1 (the root's unused sibling) gets an empty box that no walk reaches.
// slot_pre records each slot's preorder position (the tie order of the
// ordered walk).
__device__ __forceinline__ void fill_pairs(int n, int first, int stride, const lux_bvh_node* __restrict__ nodes,
                                           const uint32_t* __restrict__ pair_pos, lux_bvh_node* __restrict__ pairs,
                                           uint32_t* __restrict__ slot_pre, DevInfo* info) {
    const int node_count = 2 * n - 1;
    const int slots = 2 * n;
    for (int k = first; k < node_count; k += stride) {
        lux_bvh_node nd = nodes[k];
        const uint32_t dst = pair_pos[k];
        if (dst >= uint32_t(slots)) {
            set_error(info, kErrWalkOrder);
            continue;
        }
        if (nd.primitive_id < 0) {
            const uint32_t rc = (k + 1 < node_count) ? pair_pos[k + 1] : uint32_t(slots);
            if (rc >= uint32_t(slots)) {
                set_error(info, kErrWalkOrder);
                continue;
            }
            nd.primitive_id = ~int32_t(rc);
        }
        if (nd.escape >= 0) {
            const uint32_t e = nd.escape < node_count ? pair_pos[nd.escape] : uint32_t(slots);
            if (e >= uint32_t(slots)) {
                set_error(info, kErrWalkOrder);
                continue;
            }
            nd.escape = int32_t(e);
        }
        pairs[dst] = nd;
        slot_pre[dst] = uint32_t(k);
    }
    if (n >= 2 && first == 0) {
        lux_bvh_node pad;
        pad.bounds = box_empty();
        pad.primitive_id = -1;
        pad.escape = -1;
        pairs[1] = pad;
        slot_pre[1] = 0xffffffffu;
    }
}

// Both traversal copies of the finished node array, in one launch: the first
// `wide_blocks` workgroups make the records, the others the sibling pairs.
__global__ __launch_bounds__(kBlock) void k_copies(int n, int wide_blocks, const uint32_t* __restrict__ left,
                                                   const uint32_t* __restrict__ right,
                                                   const int32_t* __restrict__ pre_internal,
                                                   const int32_t* __restrict__ pre_leaf,
                                                   const lux_bvh_node* __restrict__ nodes,
                                                   WideNode* __restrict__ wide, int32_t* __restrict__ wide_leaf,
                                                   const uint32_t* __restrict__ pair_pos,
                                                   lux_bvh_node* __restrict__ pairs, uint32_t* __restrict__ slot_pre,
                                                   DevInfo* info) {
    const int b = int(blockIdx.x);
    if (b < wide_blocks)
        for (int i = b * kBlock + int(threadIdx.x); i < n - 1; i += wide_blocks * kBlock)
            fill_wide(n, i, left, right, pre_internal, pre_leaf, nodes, wide, wide_leaf, info);
    else
        fill_pairs(n, (b - wide_blocks) * kBlock + int(threadIdx.x), (int(gridDim.x) - wide_blocks) * kBlock, nodes,
                   pair_pos, pairs, slot_pre, info);
}

}  // namespace

// Few blocks: a block lasts as long as the climbs of one thread's leaves, so one
// leaf per thread; more blocks than the CUs hold: the climbs of four leaves in
// turn keep more of a wave's lanes at work than four waves would. Builds (with 500
// rays) at 256 / 512 / 1024 threads: 1500 triangles 140 / 122 / 114 us, 60 000 200 /
// 181 / 176, 131 072 212 / 197 / 201, 262 147 239 / 230 / 247, 400 000 282 / 283 / 319,
// 2^20 522 / 538 / 631 us. A refit has no preorder climb to share: 2^20 triangles 122
// / 107 us for the pass at 256 / 512.
template <int kMode>
void launch_local(const char* name, BvhDev& d, const lux_aabb* src_boxes, const lux_triangle* src_tris, int write_back,
                  hipStream_t s) {
    const int blocks = div_up(d.n, kLocalLeaves);
    auto go = [&](auto threads) {
        constexpr int kThreads = decltype(threads)::value;
        LUX_LAUNCH(name, (k_local<kMode, kThreads>), blocks, kThreads, 0, s, d.n, (const uint32_t*)d.vals[0],
                   (const int32_t*)d.ids, src_boxes, src_tris, d.boxes, write_back, (const uint32_t*)d.parent,
                   (const uint32_t*)d.leaf_parent, (const uint32_t*)d.first, (const uint32_t*)d.last,
                   (const uint32_t*)d.rtop_int, (const uint32_t*)d.rtop_leaf, d.nodes, d.pre_internal, d.pre_leaf,
                   d.edge_boxes, d.block_boxes, d.info);
    };
    if (blocks <= 96) {
        go(std::integral_constant<int, 1024>{});
        return;
    }
    if constexpr (kMode == 0)
        if (blocks > 384) {
            go(std::integral_constant<int, 256>{});
            return;
        }
    go(std::integral_constant<int, 512>{});
}

void wide_from(const BvhDev& d, const lux_bvh_node* nodes, WideNode* wide, int32_t* wide_leaf, hipStream_t s) {
    if (d.n < 2) return;
    const int blocks = min(4096, div_up(d.n - 1, kBlock));
    LUX_LAUNCH("lbvh_copies", k_copies, blocks, kBlock, 0, s, d.n, blocks, (const uint32_t*)d.left,
               (const uint32_t*)d.right, (const int32_t*)d.pre_internal, (const int32_t*)d.pre_leaf, nodes, wide,
               wide_leaf, (const uint32_t*)nullptr, (lux_bvh_node*)nullptr, (uint32_t*)nullptr, d.info);
}

namespace {
void launch_copies(const BvhDev& d, unsigned which, hipStream_t s) {
    if (d.n <= 0) return;
    which &= d.holds;
    const int wide_blocks = (which & kCopyRecords) && d.n > 1 ? min(4096, div_up(d.n - 1, kBlock)) : 0;
    const int pair_blocks = which & kCopyPairs ? max(1, min(2048, div_up(2 * d.n - 1, kBlock))) : 0;
    if (wide_blocks + pair_blocks == 0) return;
    LUX_LAUNCH("lbvh_copies", k_copies, wide_blocks + pair_blocks, kBlock, 0, s, d.n, wide_blocks,
               (const uint32_t*)d.left, (const uint32_t*)d.right, (const int32_t*)d.pre_internal,
               (const int32_t*)d.pre_leaf, (const lux_bvh_node*)d.nodes, d.wide, d.wide_leaf,
               (const uint32_t*)d.pair_pos, d.pairs, d.slot_pre, d.info);
}

bool capturing(hipStream_t s) {
    hipStreamCaptureStatus status = hipStreamCaptureStatusNone;
    hip_check(hipStreamIsCapturing(s, &status), "hipStreamIsCapturing");
    return status != hipStreamCaptureStatusNone;
}

// The node array has just been enqueued (build, refit).
void nodes_changed(BvhDev& d, hipStream_t s) {
    if (capturing(s)) {  // at each replay, and not yet: `stale` stays as it is
        launch_copies(d, kCopyBoth, s);
        return;
    }
    d.stale = kCopyBoth & ~d.keep;
    launch_copies(d, d.keep, s);
}
}  // namespace

void tree_copies(BvhDev& d, unsigned need, hipStream_t s) {
    const unsigned missing = d.stale & need;
    if ((d.keep & need) == need && !missing) return;
    const bool recorded = capturing(s);
    if (recorded) d.keep |= need;
    if (!missing) return;
    launch_copies(d, missing, s);
    if (!recorded) d.stale &= ~missing;
}

void keep_copies(BvhDev& d, unsigned need, hipStream_t s) {
    d.keep |= need;
    tree_copies(d, need, s);
}

void raysort_release(RaySortDev& r) {
    void* ptrs[] = {r.keys[0], r.keys[1], r.vals[0], r.vals[1], r.hist, r.status, r.tickets};
    for (void* p : ptrs)
        if (p) (void)hipFree(p);
    r = RaySortDev{};
}

size_t ray_order_status_words(int n) { return size_t(sort_tiles(n)) * kRadix; }

const uint32_t* ray_order_into(const RayOrderBufs& b, uint32_t first_epoch, const BvhDev& tree, const lux_ray* rays,
                               int n, hipStream_t s) {
    LUX_LAUNCH("ray_order_zero", k_zero_u32, 1, kBlock, 0, s, b.hist, 2 * kRadix);
    LUX_LAUNCH("ray_order_keys", k_ray_keys, max(1, min(1024, div_up(n, kBlock * 16))), kBlock, 0, s, rays, n,
               (const DevInfo*)tree.info, b.keys[0], b.vals[0], b.hist);
    const int tiles = sort_tiles(n);
    for (int p = 0; p < 2; ++p) {  // digits 14..21, then 22..29: the top 16 bits
        const int src = p & 1, dst = src ^ 1;
        LUX_LAUNCH("ray_order_sort", k_sort_pass, tiles, kBlock, 0, s, (const uint32_t*)b.keys[src],
                   (const uint32_t*)b.vals[src], b.keys[dst], b.vals[dst], n, 14 + 8 * p,
                   (const uint32_t*)(b.hist + p * kRadix), b.status, b.tickets, first_epoch + uint32_t(p), tiles,
                   tree.info);
    }
    return b.vals[0];
}

void zero_words(uint32_t* p, size_t count, hipStream_t s) {
    if (count == 0) return;
    LUX_LAUNCH("zero_words", k_zero_u32, max(1, min(1024, div_up(int64_t(count), kBlock))), kBlock, 0, s, p,
               int(count));
}

const uint32_t* ray_order(RaySortDev& r, const BvhDev& tree, const lux_ray* rays, int n, hipStream_t s) {
    if (n > r.capacity) {
        if (r.capacity) hip_check(hipDeviceSynchronize(), "synchronize before ray-sort growth");
        raysort_release(r);
        try {
            for (int b = 0; b < 2; ++b) {
                r.keys[b] = dalloc<uint32_t>(n);
                r.vals[b] = dalloc<uint32_t>(n);
            }
            r.hist = dalloc<uint32_t>(2 * kRadix);
            r.status = dalloc<uint64_t>(ray_order_status_words(n));
            r.tickets = dalloc<uint32_t>(4);
        } catch (...) {
            raysort_release(r);
            throw;
        }
        r.capacity = n;
        zero_words(reinterpret_cast<uint32_t*>(r.status), 2 * ray_order_status_words(n), s);
        zero_words(r.tickets, 4, s);
    }
    const RayOrderBufs b{{r.keys[0], r.keys[1]}, {r.vals[0], r.vals[1]}, r.hist, r.status, r.tickets};
    const uint32_t first = r.epoch + 1;
    r.epoch += 2;
    return ray_order_into(b, first, tree, rays, n, s);
}

namespace {
// Every buffer of a tree for cap primitives, with its element count.
template <typename F>
void bvh_buffers(BvhDev& d, int cap, F&& f) {
    const size_t c = size_t(cap);
    f(d.boxes, c);
    f(d.ids, c);
    for (int b = 0; b < 2; ++b) {
        f(d.keys[b], c);
        f(d.vals[b], c);
    }
    f(d.left, c);
    f(d.right, c);
    f(d.parent, c);
    f(d.first, c);
    f(d.last, c);
    f(d.leaf_parent, c);
    f(d.edge_boxes, 2 * c);
    f(d.block_boxes, size_t(div_up(cap, kLocalLeaves)));
    f(d.pre_internal, c);
    f(d.pre_leaf, c);
    f(d.nodes, 2 * c);
    f(d.rtop_int, c);
    f(d.rtop_leaf, c);
    f(d.hist, size_t(kPasses * kRadix));
    f(d.status, size_t(sort_tiles(cap)) * kRadix);
    f(d.tickets, size_t(4));
    f(d.partials, sizeof(BoxIds) * kReduceBlocksMax);
    f(d.info, size_t(1));
    f(d.counter, size_t(4));
    if (d.holds & kCopyPairs) {
        f(d.pairs, 2 * c);
        f(d.pair_pos, 2 * c);
        f(d.slot_pre, 2 * c);
    }
    if (d.holds & kCopyRecords) {
        f(d.wide, c);
        f(d.wide_leaf, 4 * c);
    }
}
}  // namespace

size_t bvh_device_bytes(int n, unsigned holds) {
    BvhDev d;
    d.holds = holds;
    size_t bytes = 0;
    bvh_buffers(d, max(n, 1), [&](auto*& p, size_t count) { bytes += sizeof(*p) * count; });
    return bytes;
}

void bvh_release(BvhDev& d) {
    bvh_buffers(d, d.capacity, [](auto*& p, size_t) {
        if (p) (void)hipFree(p);
    });
    BvhDev empty;
    d = empty;
}

void bvh_allocate(BvhDev& d, int n, hipStream_t s) {
    if (n <= d.capacity && d.info) {
        d.n = n;
        return;
    }
    const unsigned holds = d.holds, keep = d.keep;
    auto release = [&] {
        bvh_release(d);
        d.holds = holds;
        d.keep = keep;
    };
    release();
    const int cap = max(n, 1);
    d.status_words = sort_tiles(cap) * kRadix;
    try {
        bvh_buffers(d, cap, [](auto*& p, size_t count) { p = dalloc<std::remove_reference_t<decltype(*p)>>(count); });
    } catch (...) {  // a later build must not take the rest for allocated
        release();
        throw;
    }
    d.capacity = cap;
    d.n = n;
    LUX_LAUNCH("lbvh_clear", k_clear_tree, max(1, min(512, div_up(d.status_words, kBlock))), kBlock, 0, s, d.status,
               d.status_words, d.tickets, d.counter, d.info);
    d.epoch = 0;
}

namespace {
// Boxes above the leaf blocks and, in a build (layout), the pair positions.
template <bool kLayout>
void launch_top_boxes(BvhDev& d, hipStream_t s) {
    if (d.n <= kLocalLeaves) {  // one leaf block: the root is local
        if (kLayout)
            LUX_LAUNCH("lbvh_pair_layout", k_pair_layout, max(1, div_up(d.n - 1, kBlock)), kBlock, 0, s, d.n,
                       (const uint32_t*)d.left, (const uint32_t*)d.last, (const int32_t*)d.pre_internal, d.pair_pos,
                       d.info);
        return;
    }
    LUX_LAUNCH("lbvh_top_boxes", k_top_boxes<kLayout>, max(1, min(2048, div_up(d.n - 1, kBlock))), kBlock, 0, s, d.n,
               (const uint32_t*)d.first, (const uint32_t*)d.last, (const uint32_t*)d.left, d.pair_pos,
               (const int32_t*)d.pre_internal,
               (const lux_aabb*)d.edge_boxes, (const lux_aabb*)d.block_boxes, d.nodes, d.info);
}
void top_boxes(BvhDev& d, bool layout, hipStream_t s) {
    if (layout && (d.holds & kCopyPairs))
        launch_top_boxes<true>(d, s);
    else
        launch_top_boxes<false>(d, s);
}
}  // namespace

void lbvh_build(BvhDev& d, const lux_aabb* in_boxes, const int32_t* in_ids, int n, hipStream_t s) {
    bvh_allocate(d, n, s);
    if (n <= 0) return;
    int copy = (in_boxes != d.boxes || in_ids != d.ids) ? 1 : 0;
    int rb = reduce_blocks(n);
    BoxIds* partials = reinterpret_cast<BoxIds*>(d.partials);
    LUX_LAUNCH("lbvh_root_partials", k_root_partials, rb, kBlock, 0, s, in_boxes, in_ids, d.boxes, d.ids, copy,
               n, partials, d.hist, d.info);
    if (n == 1) {
        LUX_LAUNCH("lbvh_single_leaf", k_single_leaf, 1, 1, 0, s, (const lux_aabb*)d.boxes,
                   (const lux_triangle*)nullptr, (const int32_t*)d.ids, d.boxes, 0, d.nodes, d.pre_leaf,
                   d.keys[0], d.vals[0], d.info, 1);
        // root box from the one leaf (the reduction result is identical)
        top_boxes(d, true, s);
        nodes_changed(d, s);
        return;
    }
    int mh_blocks = max(1, min(1024, div_up(n, kBlock * 16)));
    LUX_LAUNCH("lbvh_morton_hist", k_morton_hist, mh_blocks, kBlock, 0, s, (const lux_aabb*)d.boxes, n,
               (const BoxIds*)partials, rb, d.info, d.keys[0], d.vals[0], d.hist);
    int tiles = sort_tiles(n);
    for (int p = 0; p < kPasses; ++p) {
        uint32_t epoch = ++d.epoch;
        int src = p & 1, dst = src ^ 1;
        LUX_LAUNCH("lbvh_sort_pass", k_sort_pass, tiles, kBlock, 0, s, (const uint32_t*)d.keys[src],
                   (const uint32_t*)d.vals[src], d.keys[dst], d.vals[dst], n, 8 * p,
                   (const uint32_t*)(d.hist + p * kRadix), d.status, d.tickets, epoch, tiles, d.info);
    }
    const int blocks = div_up(n, kLocalLeaves);
    LUX_LAUNCH("lbvh_karras", k_karras, div_up(n - 1, kBlock), kBlock, 0, s, (const uint32_t*)d.keys[0], n,
               d.left, d.right, d.parent, d.leaf_parent, d.first, d.last);
    if (blocks > 1)
        LUX_LAUNCH("lbvh_top_layout", k_top_layout, max(1, min(2048, div_up(n - 1, kBlock))), kBlock, 0, s, n,
                   (const uint32_t*)d.parent, (const uint32_t*)d.left, (const uint32_t*)d.right,
                   (const uint32_t*)d.first, (const uint32_t*)d.last, d.rtop_int, d.rtop_leaf, d.pre_internal,
                   d.info);
    launch_local<0>("lbvh_local", d, d.boxes, nullptr, 0, s);
    top_boxes(d, true, s);
    nodes_changed(d, s);
}

namespace {
template <int kMode>
void refit_launch(BvhDev& d, const lux_aabb* in_boxes, const lux_triangle* tris, hipStream_t s) {
    int n = d.n;
    int wb = (kMode == 2 || in_boxes != d.boxes) ? 1 : 0;
    if (n == 1) {
        LUX_LAUNCH("lbvh_single_leaf", k_single_leaf, 1, 1, 0, s, in_boxes, tris, (const int32_t*)d.ids, d.boxes,
                   wb, d.nodes, d.pre_leaf, d.keys[0], d.vals[0], d.info, 0);
        nodes_changed(d, s);
        return;
    }
    launch_local<kMode>(kMode == 2 ? "lbvh_local_tris" : "lbvh_local_boxes", d, in_boxes, tris, wb, s);
    top_boxes(d, false, s);
    nodes_changed(d, s);
}
}  // namespace

namespace {
// Build input from triangles (collect_scene_mesh_bvh_build_primitives,
// src/scene/scene_prepare.h:420-439): box i = triangle_bounds of triangle i
// (an empty box expanded by v0, v1, v2), id i. The triangle comes from the
// soup `tris`, or from the indexed mesh (verts, idx; indices already checked
// by the caller, a bad one leaves an empty box and sets kErrPrimRange).
__global__ __launch_bounds__(kBlock) void k_tri_input(const lux_triangle* __restrict__ tris,
                                                      const lux_vec3* __restrict__ verts,
                                                      const uint32_t* __restrict__ idx, int nv, int n,
                                                      lux_aabb* __restrict__ boxes, int32_t* __restrict__ ids,
                                                      DevInfo* info) {
    for (int i = blockIdx.x * kBlock + threadIdx.x; i < n; i += gridDim.x * kBlock) {
        lux_triangle t;
        if (tris) {
            t = tris[i];
        } else {
            const uint32_t a = idx[3 * size_t(i)], b = idx[3 * size_t(i) + 1], c = idx[3 * size_t(i) + 2];
            if (a >= uint32_t(nv) || b >= uint32_t(nv) || c >= uint32_t(nv)) {
                set_error(info, kErrPrimRange);
                boxes[i] = box_empty();
                ids[i] = i;
                continue;
            }
            t.v0 = verts[a];
            t.v1 = verts[b];
            t.v2 = verts[c];
        }
        boxes[i] = tri_box(t);
        ids[i] = i;
    }
}
}  // namespace

void lbvh_build_triangles(BvhDev& d, const lux_triangle* tris, const lux_vec3* verts, const uint32_t* idx, int nv,
                          int n, hipStream_t s) {
    bvh_allocate(d, n, s);
    if (n <= 0) return;
    LUX_LAUNCH("lbvh_tri_input", k_tri_input, std::max(1, std::min(4096, div_up(n, kBlock))), kBlock, 0, s, tris,
               verts, idx, nv, n, d.boxes, d.ids, d.info);
    lbvh_build(d, d.boxes, d.ids, n, s);
}

void lbvh_refit_boxes(BvhDev& d, const lux_aabb* in_boxes, hipStream_t s) {
    if (d.n <= 0) return;
    refit_launch<1>(d, in_boxes, nullptr, s);
}

void lbvh_refit_triangles(BvhDev& d, const lux_triangle* tris, hipStream_t s) {
    if (d.n <= 0) return;
    refit_launch<2>(d, nullptr, tris, s);
}

}  // namespace lux
