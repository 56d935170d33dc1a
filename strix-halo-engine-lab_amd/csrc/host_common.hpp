// Host side shared by the translation units: the thread's last error, argument checks, launch checks, device properties.
#pragma once
#include "mi355_strix.h"

#include <hip/hip_runtime.h>

#include <atomic>
#include <cstdint>
#include <string>

namespace strix950 {

inline thread_local std::string g_error;

inline int32_t fail(int32_t code, const char* what) {
    g_error = what;
    return code;
}
inline int32_t hip_fail(hipError_t e, const char* what) {
    g_error = std::string(what) + ": " + hipGetErrorString(e);
    return MI355_E_HIP;
}
#define STRIX_REQUIRE(cond, what) do { if (!(cond)) return fail(MI355_E_INVALID_ARGUMENT, what); } while (0)
#define STRIX_LAUNCHED(what) do { const hipError_t e_ = hipGetLastError(); if (e_ != hipSuccess) return hip_fail(e_, what); } while (0)

inline bool aligned(const void* p, size_t a) { return (reinterpret_cast<uintptr_t>(p) % a) == 0; }
inline hipStream_t hs(mi355_stream s) { return static_cast<hipStream_t>(s); }

constexpr uint32_t kQ4kBlock = 144, kQ80Block = 34;

// A property of the current device, asked once per device ordinal (0 if the runtime cannot say).
inline uint32_t device_property(hipDeviceAttribute_t what, std::atomic<uint32_t> (&known)[64]) {
    int device = 0, value = 0;
    if (hipGetDevice(&device) != hipSuccess || device < 0) return 0;
    if (device < 64) {
        const uint32_t seen = known[device].load(std::memory_order_relaxed);
        if (seen != 0) return seen;
    }
    if (hipDeviceGetAttribute(&value, what, device) != hipSuccess || value <= 0) return 0;
    if (device < 64) known[device].store(static_cast<uint32_t>(value), std::memory_order_relaxed);
    return static_cast<uint32_t>(value);
}
inline uint32_t compute_units() {
    static std::atomic<uint32_t> known[64];
    return device_property(hipDeviceAttributeMultiprocessorCount, known);
}
// LDS bytes of one compute unit
inline uint32_t lds_per_unit() {
    static std::atomic<uint32_t> known[64];
    return device_property(hipDeviceAttributeMaxSharedMemoryPerMultiprocessor, known);
}
// wavefronts of a launch that are all resident at once when each holds `lds_each` bytes of LDS
inline uint64_t resident_waves(uint32_t lds_each) {
    return static_cast<uint64_t>(compute_units()) * (lds_per_unit() / lds_each);
}

}  // namespace strix950
