// film.hip -- film output at the end of the render path: the pixel bytes of
// write_ppm (src/film/ppm.h:37-56: scale by 1/spp, Reinhard c / (1 + c), clamp
// to [0, 1], 255.999 * c^(1/2.2) truncated) and the float body of write_pfm
// (src/film/pfm.h:27-44: scale by 1/spp, rows bottom to top), from a film of
// per-pixel sums resident in HBM, and whole-file writers on top of them.
//
// The gamma step is the only one whose result the GPU's powf could change. The
// byte is floor(255.999 * powf(c, 1/2.2)), a non-decreasing function of c, so
// it is the number of thresholds t_1..t_255 at or below c, where t_k is the
// smallest float in [0, 1] whose byte is at least k. The thresholds are found
// once on the host with the host's powf (the one the reference's writer calls),
// and the kernel finds the count from a guess and the thresholds beside it. Every
// other step is a single IEEE operation, identical on both sides.
#include <cmath>
#include <cstdio>
#include <cstring>
#include <filesystem>
#include <fstream>
#include <mutex>
#include <string>
#include <vector>

#include "lux_runtime.hpp"

namespace lux {

struct PpmTable {
    float t[256];  // t[1..255]; t[0] unused
};

namespace {

constexpr int kBlock = 256;

unsigned char ppm_byte_host(float c) { return static_cast<unsigned char>(255.999f * powf(c, 1.0f / 2.2f)); }

// Smallest float in [0, 1] whose byte reaches k (bisection over the float bit
// patterns, which are ordered like the values for non-negative floats).
float threshold(int k) {
    uint32_t lo = 0, hi = 0x3f800000u;  // byte(0) = 0 < k <= 255 = byte(1)
    while (lo + 1 < hi) {
        const uint32_t mid = lo + (hi - lo) / 2;
        float c;
        std::memcpy(&c, &mid, sizeof(c));
        if (ppm_byte_host(c) >= k)
            hi = mid;
        else
            lo = mid;
    }
    float c;
    std::memcpy(&c, &hi, sizeof(c));
    return c;
}

const PpmTable& ppm_table() {
    static PpmTable table;
    static std::once_flag once;
    std::call_once(once, [] {
        table.t[0] = 0.0f;
        for (int k = 1; k < 256; ++k) table.t[k] = threshold(k);
    });
    return table;
}

// clamp01 of the reference (std::max(0, std::min(1, v))), NaN included:
// std::min(1, NaN) is 1 and std::max(0, x) keeps x unless 0 < x is false.
__device__ __forceinline__ float clamp01_ref(float v) {
    const float m = (v < 1.0f) ? v : 1.0f;
    return (0.0f < m) ? m : 0.0f;
}

// The byte of a pixel value: the count of thresholds t[1..255] at or below it. A
// guess from the hardware's log2 and exp2 (within one of the count over [0, 1]; the
// search below would also mend a worse one) is moved until t[guess] <= c <
// t[guess + 1]: two table reads in nearly every case. tab holds t[0] = 0 (c is
// never below it) and +inf behind t[255].
__device__ __forceinline__ uint32_t ppm_byte(float pixel, float inv, const float* tab) {
    float c = pixel * inv;
    c = c / (1.0f + c);
    c = clamp01_ref(c);
    const float g = 255.999f * __builtin_amdgcn_exp2f(__builtin_amdgcn_logf(c) * (1.0f / 2.2f));
    int k = int(fminf(fmaxf(g, 0.0f), 255.0f));
    while (c < tab[k]) --k;       // ends at k = 0: tab[0] = 0 <= c
    while (!(c < tab[k + 1])) ++k;  // ends at k = 255: c <= 1 < tab[256]
    return uint32_t(k);
}

// Four values a lane: one 16-byte load and one 4-byte store, the table in LDS. A
// film or byte buffer that is not aligned for that takes one value a lane. Bound by
// memory: 15 bytes a pixel, at 3840 x 2160 27 us (4.6 TB/s); 34 / 30 / 29 / 27 us
// with at most 1024 / 2048 / 4096 / 8192 workgroups; 171 us with one value a lane,
// a store a byte and an 8-step search through the kernel's arguments.
template <int kVec>
__global__ __launch_bounds__(kBlock) void k_film_ppm(const float* __restrict__ film, int64_t groups, float inv,
                                                     PpmTable tab, uint8_t* __restrict__ out) {
    __shared__ float s_tab[257];
    for (int i = threadIdx.x; i < 257; i += kBlock) s_tab[i] = i < 256 ? tab.t[i] : INFINITY;
    __syncthreads();
    for (int64_t i = int64_t(blockIdx.x) * kBlock + threadIdx.x; i < groups; i += int64_t(gridDim.x) * kBlock) {
        if constexpr (kVec == 4) {
            const float4 v = reinterpret_cast<const float4*>(film)[i];
            reinterpret_cast<uint32_t*>(out)[i] = ppm_byte(v.x, inv, s_tab) | ppm_byte(v.y, inv, s_tab) << 8 |
                                                  ppm_byte(v.z, inv, s_tab) << 16 | ppm_byte(v.w, inv, s_tab) << 24;
        } else {
            out[i] = uint8_t(ppm_byte(film[i], inv, s_tab));
        }
    }
}

__global__ __launch_bounds__(kBlock) void k_film_pfm(const float* __restrict__ film, int width, int height,
                                                     float inv, float* __restrict__ out) {
    const int64_t n = int64_t(width) * height;
    for (int64_t i = int64_t(blockIdx.x) * kBlock + threadIdx.x; i < n; i += int64_t(gridDim.x) * kBlock) {
        const int64_t y = i / width, x = i - y * width;
        const int64_t src = (int64_t(height) - 1 - y) * width + x;  // output row y is film row h-1-y
        out[3 * i] = film[3 * src] * inv;
        out[3 * i + 1] = film[3 * src + 1] * inv;
        out[3 * i + 2] = film[3 * src + 2] * inv;
    }
}

float inv_sample_count(int spp) { return spp > 0 ? 1.0f / float(spp) : 0.0f; }

int grid_for(int64_t items) { return int(std::max<int64_t>(1, std::min<int64_t>(8192, (items + kBlock - 1) / kBlock))); }

void create_parent_directories(const std::string& path) {
    std::filesystem::path parent = std::filesystem::path(path).parent_path();
    if (!parent.empty()) std::filesystem::create_directories(parent);
}

}  // namespace

void ppm_thresholds(float* out255) {
    const PpmTable& t = ppm_table();
    for (int k = 1; k < 256; ++k) out255[k - 1] = t.t[k];
}

void film_ppm(const float* film, int width, int height, int spp, uint8_t* out, hipStream_t s) {
    const int64_t pixels = int64_t(width) * height;
    if (pixels <= 0) return;
    const int64_t values = 3 * pixels;
    const bool aligned = reinterpret_cast<uintptr_t>(film) % 16 == 0 && reinterpret_cast<uintptr_t>(out) % 4 == 0;
    const int64_t quads = aligned ? values / 4 : 0;
    const float inv = inv_sample_count(spp);
    if (quads)
        LUX_LAUNCH("film_ppm", k_film_ppm<4>, grid_for(quads), kBlock, 0, s, film, quads, inv, ppm_table(), out);
    if (values > 4 * quads)  // the last one to three values, or all of them
        LUX_LAUNCH("film_ppm", k_film_ppm<1>, grid_for(values - 4 * quads), kBlock, 0, s, film + 4 * quads,
                   values - 4 * quads, inv, ppm_table(), out + 4 * quads);
}

void film_pfm(const float* film, int width, int height, int spp, float* out, hipStream_t s) {
    const int64_t pixels = int64_t(width) * height;
    if (pixels <= 0) return;
    LUX_LAUNCH("film_pfm", k_film_pfm, grid_for(pixels), kBlock, 0, s, film, width, height, inv_sample_count(spp),
               out);
}

void write_film_file(const char* path, bool ppm, const float* d_film, int width, int height, int spp, hipStream_t s) {
    const size_t pixels = size_t(width) * size_t(height);
    std::vector<char> body(ppm ? 3 * pixels : 12 * pixels);
    void* d_out = nullptr;
    if (!body.empty()) {
        hip_check(hipMalloc(&d_out, body.size()), "hipMalloc film output");
        try {
            if (ppm)
                film_ppm(d_film, width, height, spp, static_cast<uint8_t*>(d_out), s);
            else
                film_pfm(d_film, width, height, spp, static_cast<float*>(d_out), s);
            hip_check(hipMemcpyAsync(body.data(), d_out, body.size(), hipMemcpyDeviceToHost, s), "D2H film output");
            hip_check(hipStreamSynchronize(s), "synchronize");
        } catch (...) {
            (void)hipFree(d_out);
            throw;
        }
        hip_check(hipFree(d_out), "hipFree film output");
    }
    const std::string p(path);
    create_parent_directories(p);
    std::ofstream out(p, std::ios::binary);
    if (!out) throw Error(LUX_ERR_INVALID_ARGUMENT, "cannot open " + p);
    if (ppm)
        out << "P6\n" << width << " " << height << "\n255\n";
    else
        out << "PF\n" << width << " " << height << "\n-1.0\n";
    out.write(body.data(), std::streamsize(body.size()));
    if (!out) throw Error(LUX_ERR_HIP, "write failed: " + p);
}

}  // namespace lux
