// The HIP calls of libgrass_amd.so without a GPU: "device" memory is host memory (reserved, not
// touched), copies are memcpy, kernels are not run but logged.  Loaded before the library with
// RTLD_GLOBAL, so that the library's calls come here.  A test can limit the memory there is; as in HIP 7,
// a failed call stays the last error until hipGetLastError takes it, whatever succeeds in between.
#define __HIP_PLATFORM_AMD__ 1
#include <hip/hip_runtime_api.h>
#include <string.h>
#include <sys/mman.h>
#include <time.h>

#include <atomic>
#include <map>
#include <mutex>
#include <string>
#include <vector>

namespace {

std::recursive_mutex mu;
std::map<uintptr_t, size_t> live[2];  // device, pinned
size_t used[2], limit[2] = {~(size_t)0, ~(size_t)0};
hipError_t last = hipSuccess;
bool capturing = false;
std::atomic<int64_t> ahead{0};
size_t copies_in_capture = 0;
std::map<const void*, std::string> names;
std::vector<std::string> launches;
std::string joined;
struct Config {
    dim3 grid, block;
    size_t lds;
    hipStream_t s;
};
thread_local std::vector<Config> configs;

hipError_t take(int kind, void** p, size_t bytes) {
    std::lock_guard<std::recursive_mutex> lock(mu);
    *p = nullptr;
    if (bytes > limit[kind] - used[kind]) return last = hipErrorOutOfMemory;
    void* m = mmap(nullptr, bytes ? bytes : 1, PROT_READ | PROT_WRITE, MAP_PRIVATE | MAP_ANONYMOUS | MAP_NORESERVE, -1, 0);
    if (m == MAP_FAILED) return last = hipErrorOutOfMemory;
    live[kind][(uintptr_t)m] = bytes;
    used[kind] += bytes;
    *p = m;
    return hipSuccess;
}
hipError_t give(int kind, void* p) {
    std::lock_guard<std::recursive_mutex> lock(mu);
    auto it = live[kind].find((uintptr_t)p);
    if (it == live[kind].end()) return p ? last = hipErrorInvalidValue : hipSuccess;
    used[kind] -= it->second;
    munmap(p, it->second ? it->second : 1);
    live[kind].erase(it);
    return hipSuccess;
}

}  // namespace

extern "C" {

// ---- for the tests
// Device (kind 0) or pinned (1) memory: `free_bytes` more than is held now.
void fake_limit_of(int kind, size_t free_bytes) {
    std::lock_guard<std::recursive_mutex> lock(mu);
    limit[kind] = free_bytes == ~(size_t)0 ? free_bytes : used[kind] + free_bytes;
}
void fake_limit(size_t free_bytes) { fake_limit_of(0, free_bytes); }
size_t fake_used(int kind) {
    std::lock_guard<std::recursive_mutex> lock(mu);
    return used[kind];
}
// Bytes from p to the end of the device block that holds it.
size_t fake_room(uintptr_t p) {
    std::lock_guard<std::recursive_mutex> lock(mu);
    auto it = live[0].upper_bound(p);
    if (it == live[0].begin()) return 0;
    --it;
    return p < it->first + it->second ? it->first + it->second - p : 0;
}
// std::chrono::steady_clock, so many seconds ahead.
void fake_later(int seconds) { ahead += (int64_t)seconds * 1000000000; }
int64_t _ZNSt6chrono3_V212steady_clock3nowEv() {
    struct timespec t;
    clock_gettime(CLOCK_MONOTONIC, &t);
    return t.tv_sec * (int64_t)1000000000 + t.tv_nsec + ahead;
}
void fake_capturing(int on) { capturing = on; }
size_t fake_copies_in_capture() { return copies_in_capture; }
// The launches since the last call, a line each: kernel (mangled), workgroups, first 24 bytes of the first argument.
const char* fake_launches() {
    std::lock_guard<std::recursive_mutex> lock(mu);
    joined.clear();
    for (const std::string& l : launches) joined += l + "\n";
    launches.clear();
    return joined.c_str();
}

// ---- HIP
hipError_t hipMalloc(void** p, size_t bytes) { return take(0, p, bytes); }
hipError_t hipFree(void* p) { return give(0, p); }
hipError_t hipHostMalloc(void** p, size_t bytes, unsigned) { return take(1, p, bytes); }
hipError_t hipHostFree(void* p) { return give(1, p); }
hipError_t hipMemGetInfo(size_t* fr, size_t* total) {
    *total = 256ull << 30;
    *fr = *total - used[0];
    return hipSuccess;
}
hipError_t hipMemcpy(void* d, const void* s, size_t n, hipMemcpyKind) {
    memcpy(d, s, n);
    return hipSuccess;
}
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind, hipStream_t) {
    if (capturing) ++copies_in_capture;
    else memcpy(d, s, n);
    return hipSuccess;
}
hipError_t hipMemset(void* d, int v, size_t n) {
    memset(d, v, n);
    return hipSuccess;
}
hipError_t hipMemsetAsync(void* d, int v, size_t n, hipStream_t) { return hipMemset(d, v, n); }
hipError_t hipGetLastError() {
    std::lock_guard<std::recursive_mutex> lock(mu);
    const hipError_t e = last;
    last = hipSuccess;
    return e;
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
hipError_t hipDeviceGetAttribute(int* v, hipDeviceAttribute_t, int) {
    *v = 256;
    return hipSuccess;
}
hipError_t hipDeviceSynchronize() { return hipSuccess; }
hipError_t hipOccupancyMaxActiveBlocksPerMultiprocessor(int* n, const void*, int, size_t) {
    *n = 2;
    return hipSuccess;
}
hipError_t hipFuncSetAttribute(const void*, hipFuncAttribute, int) { return hipSuccess; }
hipError_t hipThreadExchangeStreamCaptureMode(hipStreamCaptureMode*) { return hipSuccess; }
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) {
    static char streams[1024];
    static size_t next = 0;
    *s = (hipStream_t)(streams + next++ % sizeof(streams));
    return hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return capturing ? last = hipErrorStreamCaptureUnsupported : hipSuccess; }
hipError_t hipStreamIsCapturing(hipStream_t, hipStreamCaptureStatus* st) {
    *st = capturing ? hipStreamCaptureStatusActive : hipStreamCaptureStatusNone;
    return hipSuccess;
}
hipError_t hipStreamWaitEvent(hipStream_t, hipEvent_t, unsigned) { return hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) {
    *e = (hipEvent_t)&capturing;
    return hipSuccess;
}
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }

void** __hipRegisterFatBinary(const void*) { return (void**)limit; }
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterFunction(void**, const void* f, char*, const char* name, unsigned, void*, void*, dim3*, dim3*, int*) {
    names[f] = name;
}
void __hipRegisterVar(void**, void*, char*, char*, int, size_t, int, int) {}
hipError_t __hipPushCallConfiguration(dim3 grid, dim3 block, size_t lds, hipStream_t s) {
    configs.push_back({grid, block, lds, s});
    return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3* grid, dim3* block, size_t* lds, hipStream_t* s) {
    const Config c = configs.back();
    configs.pop_back();
    *grid = c.grid;
    *block = c.block;
    *lds = c.lds;
    *s = c.s;
    return hipSuccess;
}
hipError_t hipLaunchKernel(const void* f, dim3 grid, dim3, void** args, size_t, hipStream_t) {
    std::lock_guard<std::recursive_mutex> lock(mu);
    uint64_t w[3];
    memcpy(w, args[0], sizeof(w));
    launches.push_back(names[f] + " " + std::to_string(grid.x) + " " + std::to_string(w[0]) + " " + std::to_string(w[1]) +
                       " " + std::to_string(w[2]));
    return hipSuccess;
}

}  // extern "C"
