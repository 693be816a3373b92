// Host-side plumbing of the C ABI: per-thread error text, launch checks, cached device facts, read-once knobs.
#pragma once
#include <hip/hip_runtime.h>
#include <stdarg.h>
#include <stdio.h>
#include <stdlib.h>
#include <atomic>
#include <string>

namespace qvb8 {
namespace host {

inline std::string& last_error() {
    static thread_local std::string msg;
    return msg;
}

inline int fail(int code, const char* fmt, ...) {
    char buf[512];
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(buf, sizeof buf, fmt, ap);
    va_end(ap);
    last_error() = buf;
    return code;
}

inline int check_launch(const char* who) {
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return fail(-3, "%s: launch failed: %s", who, hipGetErrorString(e));
    return 0;
}

// Compute units of the current device (cached per device index).
inline int device_cus() {
    static int cached[64] = {0};
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return 256;
    if (cached[dev] == 0) {
        int n = 0;
        if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n <= 0) n = 256;
        cached[dev] = n;
    }
    return cached[dev];
}

// Lets a kernel be launched with `bytes` of dynamic LDS (more than the default 64 KB); asked of the runtime once per
// kernel and device.
template <auto Kernel>
inline int raise_lds_limit(size_t bytes, const char* who) {
    static std::atomic<bool> done[64] = {};
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return fail(-3, "%s: no current device", who);
    if (!done[dev].load(std::memory_order_acquire)) {
        if (hipFuncSetAttribute((const void*)Kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes) != hipSuccess)
            return fail(-3, "%s: cannot raise the kernel's LDS limit", who);
        done[dev].store(true, std::memory_order_release);
    }
    return 0;
}

// A host that polls a word a kernel writes asks the runtime this rarely (every few hundred microseconds) whether the stream still
// runs: the question puts a marker into the stream and takes longer than most of these waits (a banded segment 59 us instead of 45).
constexpr int64_t kPollsPerQuery = 1 << 18;

// Integer knob from the environment, read on every call (cheap; lets a test change it between calls).
inline int env_int(const char* name, int dflt) {
    const char* e = getenv(name);
    return (e && *e) ? atoi(e) : dflt;
}

}  // namespace host
}  // namespace qvb8
