// Error plumbing shared by the C-ABI translation units.
#pragma once
#include <hip/hip_runtime.h>

#include <atomic>
#include <cstdarg>
#include <cstdio>

#include "../../include/verinf_hip.h"

namespace vi {

inline char *err_buf() {
    static thread_local char buf[512] = {0};
    return buf;
}

inline int fail(int code, const char *fmt, ...) {
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(err_buf(), 512, fmt, ap);
    va_end(ap);
    return code;
}

inline bool is_pow2(long long x) { return x > 0 && (x & (x - 1)) == 0; }
inline int ilog2(long long x) {
    int l = 0;
    while ((1ll << l) < x) ++l;
    return l;
}

// A workspace whose kernels use 16-byte accesses: the first such address at or behind ws.  Its *_workspace_bytes() includes
// the WS_SLACK bytes this may skip.
constexpr size_t WS_SLACK = 16;
inline void *align16(void *ws) { return (void *)(((uintptr_t)ws + 15) & ~(uintptr_t)15); }

// Waits until arrived() is true of pinned host memory that a kernel on the stream writes.  It is asked again and again (a stream
// synchronisation costs several microseconds more); every 2^16 times the stream is queried, so a failed launch or a stream that
// drained without the result ends the wait with an error instead of spinning.
template <class Arrived>
inline int wait_until(const char *who, Arrived arrived, hipStream_t s) {
    for (unsigned spins = 1;; ++spins) {
        if (arrived()) break;
        __builtin_ia32_pause();
        if ((spins & 0xFFFF) == 0) {
            hipError_t e = hipStreamQuery(s);
            if (e == hipErrorNotReady) {
                (void)hipGetLastError();                 // "not ready" is no error for the launch checks that follow
                continue;
            }
            if (e != hipSuccess) return fail(VI_EHIP, "%s: %s while waiting for a result", who, hipGetErrorString(e));
            // drained: host memory that is not coherent while a kernel runs shows the store now
            if (arrived()) break;
            return fail(VI_EHIP, "%s: the stream drained without the result", who);
        }
    }
    std::atomic_thread_fence(std::memory_order_acquire);
    return VI_OK;
}
// the same for a result behind which the kernel stores `seq`
inline int wait_for_tag(const char *who, const volatile uint64_t *flag, uint64_t seq, hipStream_t s) {
    return wait_until(who, [=] { return *flag == seq; }, s);
}

// whether the stream is being captured; the default stream cannot be, and may not be asked while another one is
inline int capturing(hipStream_t s, bool *is) {
    *is = false;
    if (!s) return VI_OK;
    hipStreamCaptureStatus status = hipStreamCaptureStatusNone;
    const hipError_t e = hipStreamIsCapturing(s, &status);
    if (e != hipSuccess) return fail(VI_EHIP, "hipStreamIsCapturing: %s", hipGetErrorString(e));
    *is = status != hipStreamCaptureStatusNone;
    return VI_OK;
}

// a tag no earlier call has used, so that nothing such a call may have left in flight can pass for this one's result
inline uint64_t new_tag() {
    static std::atomic<uint64_t> calls{0};
    return (calls.fetch_add(1) + 1) << 32;
}

}  // namespace vi

#define VI_HIP(call)                                                                      \
    do {                                                                                  \
        hipError_t e_ = (call);                                                           \
        if (e_ != hipSuccess) return vi::fail(VI_EHIP, "%s: %s", #call, hipGetErrorString(e_)); \
    } while (0)

#define VI_LAUNCH_CHECK(name)                                                             \
    do {                                                                                  \
        hipError_t e_ = hipGetLastError();                                                \
        if (e_ != hipSuccess) return vi::fail(VI_EHIP, "launch %s: %s", name, hipGetErrorString(e_)); \
    } while (0)
