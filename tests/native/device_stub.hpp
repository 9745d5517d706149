// A stand-in for the HIP runtime on the host: device memory is counted, streams and handles are checked for being
// alive, and memory given back by delete is overwritten and never reused, so that a use after it shows at once.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <new>
#include <set>

namespace stub {

[[noreturn]] inline void fail(const char* what) {
    std::fprintf(stderr, "FAILED: %s\n", what);
    std::fflush(stderr);
    std::_Exit(3);
}
inline void check(bool ok, const char* what) {
    if (!ok) fail(what);
}

inline std::map<void*, size_t> mem;  // device blocks held
inline size_t held = 0;              // their bytes
inline std::set<const void*> live;   // streams and handles

}  // namespace stub

void* operator new(size_t n) {
    char* p = static_cast<char*>(std::malloc(n + 16));
    if (!p) std::abort();
    std::memcpy(p, &n, sizeof n);
    return p + 16;
}
void operator delete(void* p) noexcept {
    if (!p) return;
    size_t n;
    std::memcpy(&n, static_cast<char*>(p) - 16, sizeof n);
    volatile unsigned char* q = static_cast<unsigned char*>(p);
    for (size_t i = 0; i < n; ++i) q[i] = 0xdd;
}
void operator delete(void* p, size_t) noexcept { operator delete(p); }

extern "C" {

hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetDeviceCount(int* n) {
    *n = 1;
    return hipSuccess;
}
hipError_t hipMemGetInfo(size_t* f, size_t* t) {
    *t = size_t(1) << 38;
    *f = *t - stub::held;
    return hipSuccess;
}
const char* hipGetErrorString(hipError_t) { return "stub"; }
hipError_t hipGetLastError() { return hipSuccess; }
hipError_t hipDeviceSynchronize() { stub::fail("hipDeviceSynchronize ends the captures of other threads"); }
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) {
    *s = reinterpret_cast<hipStream_t>(std::malloc(1));
    stub::live.insert(*s);
    return hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t s) {
    stub::check(stub::live.erase(s) == 1, "hipStreamDestroy: not a stream");
    return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t s) {
    stub::check(stub::live.count(s) == 1, "hipStreamSynchronize: not a stream");
    return hipSuccess;
}
hipError_t hipStreamQuery(hipStream_t s) {
    stub::check(stub::live.count(s) == 1, "hipStreamQuery: not a stream");
    return hipSuccess;
}

}  // extern "C"
