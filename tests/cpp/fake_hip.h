// A HIP runtime for host tests, without a GPU: a device of a given size whose memory is host memory, filled with 0xff when
// handed out; launches are recorded by kernel name and do nothing.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <new>
#include <string>
#include <vector>

namespace fake {

struct Device {
    size_t size = ~(size_t)0, live = 0;
    hipError_t last = hipSuccess;
    bool capturing = false;                                // every stream
    std::map<void*, size_t> blocks;
    std::vector<std::string> launched;
};
inline Device dev;
inline bool host_memory_gone = false;
inline std::map<const void*, std::string>& kernels() { static std::map<const void*, std::string> k; return k; }

inline int failures = 0;
inline void expect(bool ok, const char* what, unsigned long long value = 0) {
    if (!ok) { std::printf("failed: %s (%llu)\n", what, value); ++failures; }
}

struct Check { const char* name; void (*run)(); };
template <size_t N>
int run(const Check (&checks)[N], int argc, char** argv) {
    for (const Check& c : checks)
        if (argc == 2 && std::strcmp(argv[1], c.name) == 0) {
            c.run();
            if (!failures) std::printf("ok\n");
            return failures ? 1 : 0;
        }
    std::fprintf(stderr, "usage: %s <check>\n", argv[0]);
    return 2;
}

}  // namespace fake

void* operator new(size_t n) {
    void* p = fake::host_memory_gone ? nullptr : std::malloc(n ? n : 1);
    if (!p) throw std::bad_alloc();
    return p;
}
void operator delete(void* p) noexcept { std::free(p); }
void operator delete(void* p, size_t) noexcept { std::free(p); }

extern "C" {
hipError_t hipMalloc(void** p, size_t n) {
    using fake::dev;
    if (n > dev.size || dev.live + n > dev.size) return dev.last = hipErrorOutOfMemory;
    *p = std::malloc(n);
    std::memset(*p, 0xff, n);
    const bool gone = fake::host_memory_gone;              // (the map is the fake's, not the library's)
    fake::host_memory_gone = false;
    dev.blocks[*p] = n;
    fake::host_memory_gone = gone;
    dev.live += n;
    return hipSuccess;
}
hipError_t hipFree(void* p) {
    if (!p) return hipSuccess;
    fake::expect(fake::dev.blocks.count(p) == 1, "memory is freed once");
    fake::dev.live -= fake::dev.blocks[p];
    fake::dev.blocks.erase(p);
    std::free(p);
    return hipSuccess;
}
hipError_t hipMemcpy(void* to, const void* from, size_t n, hipMemcpyKind) { std::memcpy(to, from, n); return hipSuccess; }
hipError_t hipMemset(void* p, int v, size_t n) { std::memset(p, v, n); return hipSuccess; }
hipError_t hipGetDevice(int* d) { *d = 0; return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipDeviceSynchronize() { return hipSuccess; }
hipError_t hipGetLastError() { const hipError_t e = fake::dev.last; fake::dev.last = hipSuccess; return e; }
const char* hipGetErrorString(hipError_t e) { return e == hipErrorOutOfMemory ? "out of memory" : "error"; }
hipError_t hipStreamIsCapturing(hipStream_t, hipStreamCaptureStatus* s) {
    *s = fake::dev.capturing ? hipStreamCaptureStatusActive : hipStreamCaptureStatusNone;
    return hipSuccess;
}
hipError_t hipGetDevicePropertiesR0600(hipDeviceProp_tR0600* p, int) {
    std::memset(p, 0, sizeof(*p));
    p->multiProcessorCount = 256;
    return hipSuccess;
}
hipError_t hipGetSymbolAddress(void** p, const void* symbol) { *p = const_cast<void*>(symbol); return hipSuccess; }
hipError_t hipMemcpyToSymbol(const void*, const void*, size_t, size_t, hipMemcpyKind) { return hipSuccess; }
hipError_t hipMemcpyFromSymbol(void*, const void*, size_t, size_t, hipMemcpyKind) { return hipSuccess; }
hipError_t hipLaunchKernel(const void* f, dim3, dim3, void**, size_t, hipStream_t) {
    fake::dev.launched.push_back(fake::kernels()[f]);
    return hipSuccess;
}
hipError_t __hipPushCallConfiguration(dim3, dim3, size_t, hipStream_t) { return hipSuccess; }
hipError_t __hipPopCallConfiguration(dim3* grid, dim3* block, size_t* shared, hipStream_t* stream) {
    *grid = *block = dim3(1);
    *shared = 0;
    *stream = nullptr;
    return hipSuccess;
}
void** __hipRegisterFatBinary(const void*) { static void* module; return &module; }
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterFunction(void**, const void* f, char*, const char* name, unsigned, void*, void*, void*, void*, int*) {
    fake::kernels()[f] = name;
}
void __hipRegisterVar(void**, void*, char*, char*, int, size_t, int, int) {}
}
