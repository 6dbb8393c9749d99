// hip_stub.cpp - the HIP host calls that libjules_hip makes, without a GPU:
// one device, its memory from malloc (so AddressSanitizer sees every staging
// copy), launches recorded instead of run.  A launch of 2^32 threads or more
// in a dimension fails, and so does an allocation while a stream is captured
// unless the thread is in relaxed capture mode, as in the HIP runtime.
#include "hip_stub.hpp"

#include <cxxabi.h>

#include <cstdlib>
#include <cstring>
#include <mutex>

namespace stub {
std::function<void(const Launch&)> on_launch;
std::function<void(hipStream_t)> on_synchronize;
std::set<hipStream_t> capturing;

namespace {
std::mutex& mu() {
    static std::mutex m;
    return m;
}
// host address of a kernel's stub -> name; filled by static initialisers
std::map<const void*, std::string>& names() {
    static std::map<const void*, std::string> m;
    return m;
}
std::map<const char*, size_t>& blocks() {
    static std::map<const char*, size_t> m;
    return m;
}
struct Config {
    dim3 grid, block;
    size_t shared;
    hipStream_t stream;
};
thread_local Config g_config;
thread_local hipError_t g_last = hipSuccess;
thread_local hipStreamCaptureMode g_mode = hipStreamCaptureModeGlobal;

hipError_t set(hipError_t e) {
    if (e != hipSuccess) g_last = e;
    return e;
}
}  // namespace

bool allocated(const void* p) {
    std::lock_guard<std::mutex> lock(mu());
    const char* c = static_cast<const char*>(p);
    auto it = blocks().upper_bound(c);
    if (it == blocks().begin()) return false;
    --it;
    return c < it->first + it->second;
}
std::map<const char*, size_t> allocations() {
    std::lock_guard<std::mutex> lock(mu());
    return blocks();
}
}  // namespace stub

using namespace stub;

extern "C" {

extern const char __hip_fatbin[] = "";  // where the device code would be

void** __hipRegisterFatBinary(const void*) {
    static void* handle;
    return &handle;
}
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterFunction(void**, const void* host, char*, const char* name, unsigned, void*, void*, void*,
                           void*, int*) {
    int status = 0;
    char* d = abi::__cxa_demangle(name, nullptr, nullptr, &status);
    names()[host] = status == 0 ? d : name;
    std::free(d);
}
void __hipRegisterVar(void**, void*, char*, char*, int, size_t, int, int) {}
hipError_t __hipPushCallConfiguration(dim3 grid, dim3 block, size_t shared, hipStream_t stream) {
    g_config = {grid, block, shared, stream};
    return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3* grid, dim3* block, size_t* shared, hipStream_t* stream) {
    *grid = g_config.grid;
    *block = g_config.block;
    *shared = g_config.shared;
    *stream = g_config.stream;
    return hipSuccess;
}
hipError_t hipLaunchKernel(const void* f, dim3 grid, dim3 block, void** args, size_t, hipStream_t stream) {
    if (!grid.x || !grid.y || !grid.z || (uint64_t)grid.x * block.x >> 32 || (uint64_t)grid.y * block.y >> 32 ||
        (uint64_t)grid.z * block.z >> 32)
        return set(hipErrorInvalidConfiguration);
    if (on_launch) {
        const auto it = names().find(f);
        on_launch({it == names().end() ? "" : it->second, grid, block, stream, args});
    }
    return hipSuccess;
}

hipError_t hipMalloc(void** p, size_t n) {
    if (!capturing.empty() && g_mode != hipStreamCaptureModeRelaxed) return set(hipErrorStreamCaptureUnsupported);
    char* c = n >> 40 ? nullptr : static_cast<char*>(std::malloc(n ? n : 1));
    if (!c) return set(hipErrorOutOfMemory);
    std::lock_guard<std::mutex> lock(mu());
    blocks()[c] = n;
    *p = c;
    return hipSuccess;
}
hipError_t hipFree(void* p) {
    if (!p) return hipSuccess;
    {
        std::lock_guard<std::mutex> lock(mu());
        if (!blocks().erase(static_cast<char*>(p))) return set(hipErrorInvalidValue);
    }
    std::free(p);
    return hipSuccess;
}
hipError_t hipMemcpy(void* d, const void* s, size_t n, hipMemcpyKind) {
    std::memcpy(d, s, n);
    return hipSuccess;
}
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind, hipStream_t) {
    std::memcpy(d, s, n);
    return hipSuccess;
}
hipError_t hipMemcpy2D(void* d, size_t dp, const void* s, size_t sp, size_t w, size_t h, hipMemcpyKind) {
    for (size_t i = 0; i < h; ++i)
        std::memcpy(static_cast<char*>(d) + i * dp, static_cast<const char*>(s) + i * sp, w);
    return hipSuccess;
}
hipError_t hipMemset(void* d, int v, size_t n) {
    std::memset(d, v, n);
    return hipSuccess;
}
hipError_t hipPointerGetAttributes(hipPointerAttribute_t* a, const void* p) {
    if (!allocated(p)) return set(hipErrorInvalidValue);
    std::memset(a, 0, sizeof *a);
    a->type = hipMemoryTypeDevice;
    return hipSuccess;
}
hipError_t hipMemGetInfo(size_t* free_bytes, size_t* total) {
    *free_bytes = *total = size_t(1) << 38;
    return hipSuccess;
}
hipError_t hipGetSymbolAddress(void** p, const void*) {
    static char* symbol = static_cast<char*>(std::calloc(1, size_t(16) << 20));
    *p = symbol;
    return hipSuccess;
}

hipError_t hipGetDevice(int* d) {
    *d = 0;
    return hipSuccess;
}
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetDeviceCount(int* n) {
    *n = 1;
    return hipSuccess;
}
hipError_t hipGetDevicePropertiesR0600(hipDeviceProp_tR0600* p, int) {
    std::memset(p, 0, sizeof *p);
    p->multiProcessorCount = 256;
    return hipSuccess;
}
hipError_t hipGetLastError(void) {
    const hipError_t e = g_last;
    g_last = hipSuccess;
    return e;
}
const char* hipGetErrorString(hipError_t) { return "stub error"; }

hipError_t hipDeviceSynchronize(void) { return hipSuccess; }
hipError_t hipStreamCreate(hipStream_t* s) {
    *s = reinterpret_cast<hipStream_t>(std::malloc(1));
    return hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t s) {
    std::free(s);
    return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t s) {
    if (on_synchronize) on_synchronize(s);
    return hipSuccess;
}
hipError_t hipStreamIsCapturing(hipStream_t s, hipStreamCaptureStatus* st) {
    *st = capturing.count(s) ? hipStreamCaptureStatusActive : hipStreamCaptureStatusNone;
    return hipSuccess;
}
hipError_t hipThreadExchangeStreamCaptureMode(hipStreamCaptureMode* m) {
    std::swap(*m, g_mode);
    return hipSuccess;
}
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) {
    *e = reinterpret_cast<hipEvent_t>(std::malloc(1));
    return hipSuccess;
}
hipError_t hipEventDestroy(hipEvent_t e) {
    std::free(e);
    return hipSuccess;
}
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventQuery(hipEvent_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }

}  // extern "C"
