// Stands in for <hip/hip_runtime.h> where the CPU tests compile the library's
// device headers with g++: language keywords, and one wavefront's lanes as fibers.
// A lane that reaches a cross-lane operation waits there until every live lane of
// the wave has reached one; a lane that has returned takes no part (as on the
// device, where it is masked off).
#pragma once

#define __HIP_PLATFORM_AMD__ 1
#include <hip/hip_runtime_api.h>
#include <ucontext.h>

#include <bit>
#include <cmath>
#include <cstdint>
#include <cstring>
#include <functional>
#include <memory>

#undef __forceinline__
#define __forceinline__ inline
#define hipLaunchKernelGGL(...) ((void)0)

namespace simt {

constexpr int kLanes = 64;
constexpr size_t kStackBytes = 1 << 17;

struct Wave {
    ucontext_t main, ctx[kLanes];
    std::unique_ptr<char[]> stacks{new char[kLanes * kStackBytes]};
    bool live[kLanes] = {}, waiting[kLanes] = {};
    uint32_t in[kLanes] = {}, out[kLanes] = {};  // what each lane brought, and the last round's
    uint64_t took_part = 0;                      // the last round's lanes
    int lane = 0;
    std::function<void(int)> body;
};
inline Wave* wave = nullptr;

inline void lane_main() {
    wave->body(wave->lane);
    wave->live[wave->lane] = false;
    swapcontext(&wave->ctx[wave->lane], &wave->main);
}

// Runs body(lane) for lanes 0..count-1 of one wave.
inline void run(int count, std::function<void(int)> body) {
    Wave w;
    wave = &w;
    w.body = std::move(body);
    for (int i = 0; i < count; ++i) {
        getcontext(&w.ctx[i]);
        w.ctx[i].uc_stack.ss_sp = w.stacks.get() + i * kStackBytes;
        w.ctx[i].uc_stack.ss_size = kStackBytes;
        w.ctx[i].uc_link = &w.main;
        makecontext(&w.ctx[i], lane_main, 0);
        w.live[i] = true;
    }
    for (bool any = true; any;) {
        any = false;
        for (int i = 0; i < count; ++i)
            if (w.live[i] && !w.waiting[i]) {
                w.lane = i;
                swapcontext(&w.main, &w.ctx[i]);
            }
        w.took_part = 0;
        for (int i = 0; i < count; ++i)
            if (w.live[i]) {
                any = true;
                w.took_part |= uint64_t(1) << i;
                w.waiting[i] = false;
            }
        std::memcpy(w.out, w.in, sizeof(w.out));
    }
    wave = nullptr;
}

inline void meet(uint32_t x) {
    const int lane = wave->lane;
    wave->in[lane] = x;
    wave->waiting[lane] = true;
    swapcontext(&wave->ctx[lane], &wave->main);
}

}  // namespace simt

inline uint64_t __ballot(int p) {
    simt::meet(p ? 1u : 0u);
    uint64_t m = 0;
    for (int i = 0; i < simt::kLanes; ++i)
        if ((simt::wave->took_part >> i & 1) && simt::wave->out[i]) m |= uint64_t(1) << i;
    return m;
}
template <typename T>
inline T __shfl(T v, int src, int = 64) {
    static_assert(sizeof(T) == 4);
    simt::meet(std::bit_cast<uint32_t>(v));
    return std::bit_cast<T>(simt::wave->out[src & 63]);
}
template <typename T>
inline T __shfl_xor(T v, int mask, int = 64) {
    static_assert(sizeof(T) == 4);
    const int lane = simt::wave->lane;
    simt::meet(std::bit_cast<uint32_t>(v));
    return std::bit_cast<T>(simt::wave->out[lane ^ mask]);
}
inline int __builtin_amdgcn_readfirstlane(int v) {
    simt::meet(uint32_t(v));
    return int(simt::wave->out[std::countr_zero(simt::wave->took_part)]);
}
inline uint32_t __lane_id() { return uint32_t(simt::wave->lane); }
inline int __popcll(unsigned long long x) { return std::popcount(x); }
inline int __ffs(int x) { return __builtin_ffs(x); }
inline int __ffsll(unsigned long long x) { return __builtin_ffsll((long long)x); }
inline float __uint_as_float(uint32_t x) { return std::bit_cast<float>(x); }
inline uint32_t __float_as_uint(float x) { return std::bit_cast<uint32_t>(x); }
inline int __float_as_int(float x) { return std::bit_cast<int>(x); }
inline float __int_as_float(int x) { return std::bit_cast<float>(x); }
inline float __builtin_amdgcn_rcpf(float x) { return 1.0f / x; }

#define __HIP_MEMORY_SCOPE_AGENT 0
template <typename T, typename U>
inline T __hip_atomic_fetch_add(T* p, U v, int, int) {
    const T old = *p;
    *p = T(old + v);
    return old;
}
template <typename T, typename U>
inline T __hip_atomic_fetch_or(T* p, U v, int, int) {
    const T old = *p;
    *p = T(old | v);
    return old;
}
struct SimtIndex {
    uint32_t x = 0;
};
inline SimtIndex gridDim{1}, blockIdx, threadIdx;
