// hip_stub.cpp -- a stand-in for the HIP runtime, so that the library's host
// code (liblux_hip.so) can be stepped on the CPU: device memory is host memory,
// kernels do not run (a callback sees each launch), copies happen at once.
//
// What a real device leaves open is made as bad as it may be: memory from
// hipMalloc holds old bytes, and a fill by hipMemset, which is ordered on the
// null stream alone and returns before it is done, stays pending until the
// device is waited for. (The library's streams are non-blocking: nothing orders
// the null stream before them.)
//
// Loaded with RTLD_GLOBAL before liblux_hip.so, whose hip* symbols then resolve
// to these.
#define __HIP_PLATFORM_AMD__ 1
#include <hip/hip_runtime_api.h>

#include <cstdint>
#include <cstdlib>
#include <cstring>
#include <map>
#include <mutex>
#include <string>
#include <vector>

namespace {

struct Fill {
    void* p;
    int value;
    size_t bytes;
};

std::recursive_mutex g_mu;
std::map<const void*, std::string> g_names;   // kernel -> mangled name
std::map<const void*, size_t> g_live;         // device allocations
std::map<const void*, void*> g_symbols;       // __device__ variables
std::map<const void*, size_t> g_symbol_bytes;
std::map<void*, long> g_launches, g_waited;   // per stream: launches and copies so far, and when it was last waited for
std::vector<Fill> g_pending;                  // null-stream fills not yet done
size_t g_live_bytes = 0;
int g_null_writes = 0;                        // device writes ordered on the null stream only
int g_next = 1;
bool g_capturing = false;
int g_allocs_left = -1;  // allocations until one fails (-1: none does)
using LaunchCb = void (*)(const char* name, void* stream, void** args);
LaunchCb g_on_launch = nullptr;
using DownloadCb = void (*)(void* stream);
DownloadCb g_on_download = nullptr;  // before each asynchronous copy to the host

struct Config {
    dim3 grid, block;
    size_t shmem;
    hipStream_t stream;
};
thread_local Config t_cfg;
thread_local unsigned t_grid = 0, t_block = 0;  // of the launch the callback sees

template <typename T>
T handle() {
    return reinterpret_cast<T>(uintptr_t(0x1000) * uintptr_t(g_next++));
}

void finish_fills() {
    for (const Fill& f : g_pending) std::memset(f.p, f.value, f.bytes);
    g_pending.clear();
}

void drop_fills(const void* p, size_t bytes) {
    std::vector<Fill> keep;
    for (const Fill& f : g_pending)
        if (f.p < p || f.p >= static_cast<const char*>(p) + bytes) keep.push_back(f);
    g_pending = keep;
}

}  // namespace

extern "C" {

void stub_on_launch(LaunchCb cb) { g_on_launch = cb; }
void stub_on_download(DownloadCb cb) { g_on_download = cb; }
uint64_t stub_live_bytes() { return g_live_bytes; }
int stub_null_writes() { return g_null_writes; }
long stub_launches(void* s) {
    std::lock_guard<std::recursive_mutex> lk(g_mu);
    return g_launches[s];
}
long stub_waited(void* s) {
    std::lock_guard<std::recursive_mutex> lk(g_mu);
    return g_waited[s];
}
unsigned stub_grid() { return t_grid; }
unsigned stub_block() { return t_block; }
void stub_capturing(int on) { g_capturing = on != 0; }
void stub_fail_alloc_after(int count) { g_allocs_left = count; }

// ---- kernels ----
void** __hipRegisterFatBinary(const void*) {
    static void* module = nullptr;
    return &module;
}
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterFunction(void**, const void* host, char*, const char* name, unsigned, void*, void*, void*, void*,
                           int*) {
    g_names[host] = name;
}
void __hipRegisterVar(void**, void* var, char*, char*, int, size_t bytes, int, int) { g_symbol_bytes[var] = bytes; }
hipError_t __hipPushCallConfiguration(dim3 grid, dim3 block, size_t shmem, hipStream_t stream) {
    t_cfg = Config{grid, block, shmem, stream};
    return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3* grid, dim3* block, size_t* shmem, hipStream_t* stream) {
    *grid = t_cfg.grid;
    *block = t_cfg.block;
    *shmem = t_cfg.shmem;
    *stream = t_cfg.stream;
    return hipSuccess;
}
hipError_t hipLaunchKernel(const void* fn, dim3 grid, dim3 block, void** args, size_t, hipStream_t stream) {
    std::string name;
    {
        std::lock_guard<std::recursive_mutex> lk(g_mu);
        name = g_names.count(fn) ? g_names[fn] : "?";
        if (!stream) ++g_null_writes;
        ++g_launches[stream];
    }
    t_grid = grid.x;
    t_block = block.x;
    if (g_on_launch) g_on_launch(name.c_str(), stream, args);
    return hipSuccess;
}

// ---- memory ----
hipError_t hipMalloc(void** p, size_t bytes) {
    std::lock_guard<std::recursive_mutex> lk(g_mu);
    if (g_allocs_left == 0) return hipErrorOutOfMemory;
    if (g_allocs_left > 0) --g_allocs_left;
    *p = std::aligned_alloc(4096, (bytes + 4095) / 4096 * 4096);
    if (!*p) return hipErrorOutOfMemory;
    // old bytes: words of 1, so that a look-back word reads as epoch 1
    if (bytes <= (size_t(64) << 20))
        for (size_t i = 0; i + 4 <= bytes; i += 4) reinterpret_cast<uint32_t*>(*p)[i / 4] = 1u;
    g_live[*p] = bytes;
    g_live_bytes += bytes;
    return hipSuccess;
}
hipError_t hipFree(void* p) {
    std::lock_guard<std::recursive_mutex> lk(g_mu);
    finish_fills();  // waits for the device
    auto it = g_live.find(p);
    if (it == g_live.end()) return p ? hipErrorInvalidValue : hipSuccess;
    g_live_bytes -= it->second;
    drop_fills(p, it->second);
    g_live.erase(it);
    std::free(p);
    return hipSuccess;
}
hipError_t hipHostMalloc(void** p, size_t bytes, unsigned) {
    *p = std::calloc(1, bytes);
    return hipSuccess;
}
hipError_t hipHostFree(void* p) {
    std::free(p);
    return hipSuccess;
}
hipError_t hipMemset(void* p, int value, size_t bytes) {
    std::lock_guard<std::recursive_mutex> lk(g_mu);
    ++g_null_writes;
    g_pending.push_back(Fill{p, value, bytes});
    return hipSuccess;
}
hipError_t hipMemcpy(void* dst, const void* src, size_t bytes, hipMemcpyKind kind) {
    std::lock_guard<std::recursive_mutex> lk(g_mu);
    if (kind != hipMemcpyDeviceToHost) ++g_null_writes;
    std::memcpy(dst, src, bytes);
    return hipSuccess;
}
hipError_t hipMemcpyAsync(void* dst, const void* src, size_t bytes, hipMemcpyKind kind, hipStream_t s) {
    if (kind == hipMemcpyDeviceToHost && g_on_download) g_on_download(s);
    std::lock_guard<std::recursive_mutex> lk(g_mu);
    ++g_launches[s];
    if (!s && kind != hipMemcpyDeviceToHost) ++g_null_writes;
    std::memcpy(dst, src, bytes);
    return hipSuccess;
}
hipError_t hipGetSymbolAddress(void** p, const void* symbol) {
    std::lock_guard<std::recursive_mutex> lk(g_mu);
    void*& a = g_symbols[symbol];
    if (!a) a = std::aligned_alloc(4096, (g_symbol_bytes[symbol] + 4095) / 4096 * 4096);
    *p = a;
    return hipSuccess;
}

// ---- streams, events, graphs, device ----
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned flags) {
    if (flags != hipStreamNonBlocking) return hipErrorInvalidValue;
    *s = handle<hipStream_t>();
    return hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t s) {  // that stream's work; fills stay pending
    std::lock_guard<std::recursive_mutex> lk(g_mu);
    g_waited[s] = g_launches[s];
    return hipSuccess;
}
hipError_t hipDeviceSynchronize() {
    std::lock_guard<std::recursive_mutex> lk(g_mu);
    finish_fills();
    g_waited = g_launches;
    return hipSuccess;
}
hipError_t hipEventCreate(hipEvent_t* e) {
    *e = handle<hipEvent_t>();
    return hipSuccess;
}
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) { return hipEventCreate(e); }
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventQuery(hipEvent_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float* ms, hipEvent_t, hipEvent_t) {
    *ms = 0;
    return hipSuccess;
}
hipError_t hipStreamIsCapturing(hipStream_t, hipStreamCaptureStatus* status) {
    *status = g_capturing ? hipStreamCaptureStatusActive : hipStreamCaptureStatusNone;
    return hipSuccess;
}
hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) { return hipErrorNotSupported; }
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t*) { return hipErrorNotSupported; }
hipError_t hipGraphInstantiate(hipGraphExec_t*, hipGraph_t, hipGraphNode_t*, char*, size_t) {
    return hipErrorNotSupported;
}
hipError_t hipGraphLaunch(hipGraphExec_t, hipStream_t) { return hipErrorNotSupported; }
hipError_t hipGraphDestroy(hipGraph_t) { return hipSuccess; }
hipError_t hipGraphExecDestroy(hipGraphExec_t) { return hipSuccess; }
hipError_t hipGetDeviceCount(int* n) {
    *n = 1;
    return hipSuccess;
}
hipError_t hipGetDevice(int* d) {
    *d = 0;
    return hipSuccess;
}
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipDeviceGetAttribute(int* v, hipDeviceAttribute_t, int) {
    *v = 256;
    return hipSuccess;
}
hipError_t hipGetDevicePropertiesR0600(hipDeviceProp_tR0600* p, int) {
    std::memset(p, 0, sizeof(*p));
    return hipSuccess;
}
hipError_t hipOccupancyMaxActiveBlocksPerMultiprocessor(int* n, const void*, int, size_t) {
    *n = 2;
    return hipSuccess;
}
hipError_t hipGetLastError() { return hipSuccess; }
const char* hipGetErrorString(hipError_t) { return "stub error"; }

}  // extern "C"
