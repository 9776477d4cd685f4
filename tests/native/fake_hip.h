// A HIP runtime of host memory for the test programs: two devices with a limit on their memory, streams
// that count the work queued and not waited for, and a launch that can be made to fail.  Kernels do
// nothing.  The program defines the functions libhv.so calls, so the library's own references bind
// to them.
#pragma once
#include <hip/hip_runtime.h>
#include <atomic>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <mutex>
#include <vector>

namespace fake {
struct Block {
    size_t n;
    int device;
};
struct State {
    std::mutex mu;
    std::map<void*, Block> device, host;
    size_t used[2] = {0, 0}, limit[2] = {(size_t)1 << 40, (size_t)1 << 40};
    std::map<hipStream_t, int> queued;          // work not waited for
    std::map<hipStream_t, int> stream_device;   // of the streams made here
    std::vector<int> copy_device;               // the current device at each copy
    int launches = 0, fail_at = -1;             // the launch of this number fails
};
inline State& S() {
    static State* s = new State();
    return *s;
}
inline thread_local int current = 0;
inline thread_local hipError_t last = hipSuccess;
inline hipError_t fail(hipError_t e) {
    last = e;
    return e;
}
inline void queue(hipStream_t st) {
    std::lock_guard<std::mutex> lk(S().mu);
    ++S().queued[st];
}
inline int waiting() {
    std::lock_guard<std::mutex> lk(S().mu);
    int n = 0;
    for (auto& kv : S().queued) n += kv.second;
    return n;
}
}  // namespace fake

extern "C" {
void** __hipRegisterFatBinary(const void*) {
    static void* h = nullptr;
    return &h;
}
void __hipRegisterFunction(void**, const void*, char*, const char*, unsigned, void*, void*, void*, void*, int*) {}
void __hipRegisterVar(void**, void*, char*, char*, int, size_t, int, int) {}
void __hipUnregisterFatBinary(void**) {}
static thread_local struct {
    dim3 g, b;
    size_t sh;
    hipStream_t st;
} fake_call;
hipError_t __hipPushCallConfiguration(dim3 g, dim3 b, size_t sh, hipStream_t st) {
    fake_call = {g, b, sh, st};
    return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3* g, dim3* b, size_t* sh, hipStream_t* st) {
    *g = fake_call.g;
    *b = fake_call.b;
    *sh = fake_call.sh;
    *st = fake_call.st;
    return hipSuccess;
}
hipError_t hipLaunchKernel(const void*, dim3, dim3, void**, size_t, hipStream_t st) {
    {
        std::lock_guard<std::mutex> lk(fake::S().mu);
        if (fake::S().launches++ == fake::S().fail_at) return fake::fail(hipErrorLaunchFailure);
    }
    fake::queue(st);
    return hipSuccess;
}
hipError_t hipGetDeviceCount(int* n) {
    *n = 2;
    return hipSuccess;
}
hipError_t hipSetDevice(int d) {
    if (d < 0 || d > 1) return fake::fail(hipErrorInvalidDevice);
    fake::current = d;
    return hipSuccess;
}
hipError_t hipGetDevice(int* d) {
    *d = fake::current;
    return hipSuccess;
}
hipError_t hipDeviceGetAttribute(int* v, hipDeviceAttribute_t, int) {
    *v = 64;
    return hipSuccess;
}
hipError_t hipGetDevicePropertiesR0600(hipDeviceProp_tR0600* p, int) {
    std::memset(p, 0, sizeof *p);
    std::strcpy(p->gcnArchName, "gfx950");
    p->warpSize = 64;
    p->multiProcessorCount = 256;
    p->maxThreadsPerBlock = 1024;
    return hipSuccess;
}
int hipGetStreamDeviceId(hipStream_t st) {
    std::lock_guard<std::mutex> lk(fake::S().mu);
    auto it = fake::S().stream_device.find(st);
    return it == fake::S().stream_device.end() ? fake::current : it->second;
}
hipError_t hipGetLastError() {
    const hipError_t e = fake::last;
    fake::last = hipSuccess;
    return e;
}
const char* hipGetErrorString(hipError_t) { return "fake error"; }
hipError_t hipGetSymbolAddress(void** p, const void*) {
    static char* mem = (char*)std::calloc(1, (size_t)256 << 20);
    *p = mem;
    return hipSuccess;
}
hipError_t hipMalloc(void** p, size_t n) {
    auto& s = fake::S();
    std::lock_guard<std::mutex> lk(s.mu);
    if (s.used[fake::current] + n > s.limit[fake::current]) return fake::fail(hipErrorOutOfMemory);
    *p = std::calloc(1, n);
    s.device[*p] = {n, fake::current};
    s.used[fake::current] += n;
    return hipSuccess;
}
hipError_t hipFree(void* p) {
    auto& s = fake::S();
    std::lock_guard<std::mutex> lk(s.mu);
    auto it = s.device.find(p);
    if (it == s.device.end()) return p ? fake::fail(hipErrorInvalidValue) : hipSuccess;
    s.used[it->second.device] -= it->second.n;
    s.device.erase(it);
    for (auto& kv : s.queued) kv.second = 0;   // it waits for the device
    std::free(p);
    return hipSuccess;
}
hipError_t hipHostMalloc(void** p, size_t n, unsigned) {
    std::lock_guard<std::mutex> lk(fake::S().mu);
    *p = std::calloc(1, n);
    fake::S().host[*p] = {n, fake::current};
    return hipSuccess;
}
hipError_t hipHostFree(void* p) {
    std::lock_guard<std::mutex> lk(fake::S().mu);
    fake::S().host.erase(p);
    std::free(p);
    return hipSuccess;
}
hipError_t hipMemcpy(void* d, const void* s, size_t n, hipMemcpyKind) {
    std::memcpy(d, s, n);
    return hipSuccess;
}
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind, hipStream_t st) {
    std::memcpy(d, s, n);
    fake::queue(st);
    std::lock_guard<std::mutex> lk(fake::S().mu);
    fake::S().copy_device.push_back(fake::current);
    return hipSuccess;
}
hipError_t hipMemsetAsync(void* d, int v, size_t n, hipStream_t st) {
    std::memset(d, v, n);
    fake::queue(st);
    return hipSuccess;
}
hipError_t hipMemsetD32Async(hipDeviceptr_t d, int v, size_t n, hipStream_t st) {
    for (size_t i = 0; i < n; ++i) ((int*)d)[i] = v;
    fake::queue(st);
    return hipSuccess;
}
hipError_t hipStreamCreateWithFlags(hipStream_t* st, unsigned) {
    std::lock_guard<std::mutex> lk(fake::S().mu);
    *st = (hipStream_t)std::malloc(16);
    fake::S().stream_device[*st] = fake::current;
    return hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t st) {
    std::lock_guard<std::mutex> lk(fake::S().mu);
    fake::S().queued.erase(st);
    fake::S().stream_device.erase(st);
    std::free(st);
    return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t st) {
    std::lock_guard<std::mutex> lk(fake::S().mu);
    fake::S().queued[st] = 0;
    return hipSuccess;
}
hipError_t hipStreamWaitEvent(hipStream_t, hipEvent_t, unsigned) { return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t* e) {
    *e = (hipEvent_t)std::malloc(16);
    return hipSuccess;
}
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) { return hipEventCreate(e); }
hipError_t hipEventDestroy(hipEvent_t e) {
    std::free(e);
    return hipSuccess;
}
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float* ms, hipEvent_t, hipEvent_t) {
    *ms = 0.f;
    return hipSuccess;
}
}  // extern "C"
