// hip_on_host.h -- the part of the HIP runtime that libcismgpu.so calls, on
// host memory and without kernels, for CPU tests of the library's host code:
// allocation failures, copies, and which kernels a call would launch.  The
// program that includes it exports these symbols (-rdynamic), so the library
// it loads binds to them.  A launch runs nothing; its kernel's mangled name
// is kept, and on_launch, when set, sees the name and the arguments.
#pragma once
#include <hip/hip_runtime_api.h>

#include <atomic>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <functional>
#include <map>
#include <mutex>
#include <new>
#include <string>
#include <vector>

namespace onhost {

inline std::map<const void*, std::string> kernels;
inline std::vector<std::string> launched;
inline dim3 grid;                         // of the last launch
inline std::function<void(const std::string&, void**)> on_launch;
inline std::atomic<bool> heap_fails{false};   // operator new throws
inline bool fail_malloc = false;          // hipMalloc fails
inline bool fail_pinned = false;          // hipHostMalloc fails
inline long long copies_to_failure = -1;  // >= 0: so many more copies succeed
inline hipError_t last = hipSuccess;
inline std::mutex mtx;

inline hipError_t set(hipError_t e) {
    if (e != hipSuccess) last = e;
    return e;
}
inline bool copy_fails() {
    std::lock_guard<std::mutex> g(mtx);
    if (copies_to_failure < 0) return false;
    if (copies_to_failure == 0) return true;
    --copies_to_failure;
    return false;
}
inline int count(const char* part) {      // launches of kernels whose name contains part
    int n = 0;
    for (const auto& k : launched) n += k.find(part) != std::string::npos;
    return n;
}

struct Config { dim3 grid, block; size_t lds; hipStream_t s; };
inline thread_local Config config;

}  // namespace onhost

void* operator new(size_t n) {
    void* p = onhost::heap_fails ? nullptr : malloc(n ? n : 1);
    if (!p) throw std::bad_alloc();
    return p;
}
void operator delete(void* p) noexcept { free(p); }
void operator delete(void* p, size_t) noexcept { free(p); }

extern "C" {
void** __hipRegisterFatBinary(const void*) {
    static void* h = nullptr;
    return &h;
}
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterFunction(void**, const void* host, char*, const char* name, unsigned, void*, void*, void*, void*, int*) {
    onhost::kernels[host] = name;
}
void __hipRegisterVar(void**, void*, char*, char*, int, size_t, int, int) {}
hipError_t __hipPushCallConfiguration(dim3 g, dim3 b, size_t lds, hipStream_t s) {
    onhost::config = {g, b, lds, s};
    return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3* g, dim3* b, size_t* lds, hipStream_t* s) {
    *g = onhost::config.grid; *b = onhost::config.block; *lds = onhost::config.lds; *s = onhost::config.s;
    return hipSuccess;
}
hipError_t hipLaunchKernel(const void* f, dim3 g, dim3, void** args, size_t, hipStream_t) {
    const std::string& name = onhost::kernels[f];
    if (!onhost::heap_fails) onhost::launched.push_back(name);
    onhost::grid = g;
    if (onhost::on_launch) onhost::on_launch(name, args);
    return hipSuccess;
}

hipError_t hipMalloc(void** p, size_t n) {
    *p = onhost::fail_malloc ? nullptr : calloc(n ? n : 1, 1);
    return onhost::set(*p ? hipSuccess : hipErrorOutOfMemory);
}
hipError_t hipFree(void* p) { free(p); return hipSuccess; }
hipError_t hipHostMalloc(void** p, size_t n, unsigned) {
    *p = onhost::fail_pinned ? nullptr : calloc(n ? n : 1, 1);
    return onhost::set(*p ? hipSuccess : hipErrorOutOfMemory);
}
hipError_t hipHostFree(void* p) { free(p); return hipSuccess; }
hipError_t hipMemcpy(void* d, const void* s, size_t n, hipMemcpyKind) {
    if (onhost::copy_fails()) return onhost::set(hipErrorUnknown);
    memcpy(d, s, n);
    return hipSuccess;
}
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind k, hipStream_t) { return hipMemcpy(d, s, n, k); }
hipError_t hipMemsetAsync(void* d, int v, size_t n, hipStream_t) { memset(d, v, n); return hipSuccess; }
hipError_t hipMemcpyToSymbol(const void*, const void*, size_t, size_t, hipMemcpyKind) { return hipSuccess; }
hipError_t hipGetSymbolAddress(void** p, const void* s) { *p = const_cast<void*>(s); return hipSuccess; }

hipError_t hipGetDevice(int* d) { *d = 0; return hipSuccess; }
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetDeviceCount(int* n) { *n = 1; return hipSuccess; }
hipError_t hipDeviceGetAttribute(int* v, hipDeviceAttribute_t, int) { *v = 256; return hipSuccess; }
const char* hipGetErrorString(hipError_t e) { return e == hipSuccess ? "no error" : "error"; }
hipError_t hipGetLastError(void) {
    const hipError_t e = onhost::last;
    onhost::last = hipSuccess;
    return e;
}

hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) { *s = nullptr; return hipSuccess; }
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipStreamQuery(hipStream_t) { return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t* e) { *e = (hipEvent_t)&onhost::mtx; return hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) { return hipEventCreate(e); }
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float* ms, hipEvent_t, hipEvent_t) { *ms = 0.f; return hipSuccess; }
}
