// A host-only stand-in for the few HIP calls of device_memory.hpp: devices of `capacity` bytes together, whose
// blocks are host addresses, and a capture on some other stream that an unguarded allocation breaks.
#pragma once

#include <cstddef>
#include <cstdint>
#include <functional>
#include <map>

enum hipError_t { hipSuccess = 0, hipErrorOutOfMemory = 2, hipErrorUnknown = 999, hipErrorStreamCaptureUnsupported = 900 };
enum hipStreamCaptureMode { hipStreamCaptureModeGlobal, hipStreamCaptureModeThreadLocal, hipStreamCaptureModeRelaxed };

namespace stub {
inline size_t capacity = 1600, used = 0, frees = 0, mallocs = 0;
inline uintptr_t next = 0x1000;
inline int device = 0;
inline std::map<void*, size_t> live;
inline bool capturing = false, broken = false, fail_next = false;
inline hipStreamCaptureMode mode = hipStreamCaptureModeGlobal;
inline std::function<void()> during_malloc;  // run once, inside the next hipMalloc
}  // namespace stub

inline hipError_t hipMalloc(void** p, size_t bytes) {
    ++stub::mallocs;
    if (stub::during_malloc) {
        const std::function<void()> hook = std::move(stub::during_malloc);
        stub::during_malloc = nullptr;
        hook();
    }
    if (stub::capturing && stub::mode != hipStreamCaptureModeRelaxed) {
        stub::broken = true;
        return hipErrorStreamCaptureUnsupported;
    }
    if (stub::fail_next) {
        stub::fail_next = false;
        return hipErrorUnknown;
    }
    if (bytes > stub::capacity - stub::used) return hipErrorOutOfMemory;
    stub::used += bytes;
    *p = reinterpret_cast<void*>(stub::next += 0x1000);
    stub::live[*p] = bytes;
    return hipSuccess;
}
inline hipError_t hipFree(void* p) {
    ++stub::frees;
    stub::used -= stub::live.at(p);
    stub::live.erase(p);
    return hipSuccess;
}
inline hipError_t hipGetDevice(int* d) { return *d = stub::device, hipSuccess; }
inline hipError_t hipSetDevice(int d) { return stub::device = d, hipSuccess; }
inline hipError_t hipDeviceTotalMem(size_t* total, int) { return *total = stub::capacity, hipSuccess; }
inline hipError_t hipGetLastError() { return hipSuccess; }
inline const char* hipGetErrorString(hipError_t) { return "stub"; }
inline hipError_t hipThreadExchangeStreamCaptureMode(hipStreamCaptureMode* m) {
    const hipStreamCaptureMode before = stub::mode;
    stub::mode = *m;
    *m = before;
    return hipSuccess;
}
