// A HIP runtime for tests of the library's host code without a device: the program
// defines the runtime calls that the entry points make, and the library, linked to it,
// binds to these.  Kernels do not run: a launch is checked against the device's limits
// and recorded.  As in the runtime, an error stays pending until hipGetLastError.
#pragma once

#define __HIP_PLATFORM_AMD__ 1
#include <hip/hip_runtime.h>

#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <map>
#include <string>
#include <vector>

namespace fake {
struct Launch {
    std::string kernel;  // mangled
    dim3 grid, block;
    int arg2;  // the third argument, for kernels whose third is an int
};
// kernels by the host address that launches name; filled while the library is loaded
inline std::map<const void*, std::string>& kernels() {
    static std::map<const void*, std::string> k;
    return k;
}
inline hipError_t pending = hipSuccess;
inline size_t memory = ~(size_t)0;  // what one allocation can get
inline std::vector<size_t> asked;   // sizes of the allocations, also of those that failed
inline std::vector<Launch> launches;
inline dim3 next_grid, next_block;
inline size_t next_lds;
inline hipStream_t next_stream;

inline hipError_t fail(hipError_t e) { return pending = e; }
inline void reset() {
    pending = hipSuccess;
    memory = ~(size_t)0;
    asked.clear();
    launches.clear();
}
}  // namespace fake

#undef hipGetDevice
#undef hipMallocFromPoolAsync
extern "C" {
void** __hipRegisterFatBinary(const void*) {
    static void* module;
    return &module;
}
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterVar(void**, void*, char*, char*, int, size_t, int, int) {}
void __hipRegisterFunction(void**, const void* host, char*, const char* name, unsigned, void*, void*, void*, void*, int*) {
    fake::kernels()[host] = name;
}
hipError_t hipGetDevice(int* d) { return *d = 0, hipSuccess; }
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetLastError() {
    const hipError_t e = fake::pending;
    fake::pending = hipSuccess;
    return e;
}
hipError_t hipDeviceGetAttribute(int* v, hipDeviceAttribute_t, int) { return *v = 256, hipSuccess; }
hipError_t hipDeviceSynchronize() { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipStreamIsCapturing(hipStream_t, hipStreamCaptureStatus* s) {
    return *s = hipStreamCaptureStatusNone, hipSuccess;
}
hipError_t hipMemPoolCreate(hipMemPool_t* p, const hipMemPoolProps*) { return *p = nullptr, hipSuccess; }
hipError_t hipMemPoolSetAttribute(hipMemPool_t, hipMemPoolAttr, void*) { return hipSuccess; }
hipError_t hipMallocFromPoolAsync(void** p, size_t bytes, hipMemPool_t, hipStream_t) {
    static uintptr_t next = 1ull << 40;  // addresses that nothing reads
    fake::asked.push_back(bytes);
    if (bytes > fake::memory) return fake::fail(hipErrorOutOfMemory);
    *p = reinterpret_cast<void*>(next);
    next += (bytes + 255) & ~(size_t)255;
    return hipSuccess;
}
hipError_t hipFreeAsync(void*, hipStream_t) { return hipSuccess; }
hipError_t __hipPushCallConfiguration(dim3 grid, dim3 block, size_t lds, hipStream_t s) {
    fake::next_grid = grid, fake::next_block = block, fake::next_lds = lds, fake::next_stream = s;
    return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3* grid, dim3* block, size_t* lds, hipStream_t* s) {
    *grid = fake::next_grid, *block = fake::next_block, *lds = fake::next_lds, *s = fake::next_stream;
    return hipSuccess;
}
hipError_t hipLaunchKernel(const void* f, dim3 grid, dim3 block, void** args, size_t, hipStream_t) {
    const dim3 g = grid, b = block;
    const uint64_t x = (uint64_t)g.x * b.x, y = (uint64_t)g.y * b.y, z = (uint64_t)g.z * b.z;
    if (!x || !y || !z) return fake::fail(hipErrorInvalidConfiguration);
    if (x > UINT32_MAX || y > UINT32_MAX || z > UINT32_MAX || g.y > 65535 || g.z > 65535 ||
        (uint64_t)b.x * b.y * b.z > 1024)
        return fake::fail(hipErrorInvalidConfiguration);
    const std::string& name = fake::kernels()[f];
    fake::launches.push_back({name, g, b, name.find("k_vcsr_find_long") != std::string::npos ? *(const int*)args[2] : 0});
    return hipSuccess;
}
}
