// Memory that a handle allocates when a call first wants it, and does without where there is none.
#pragma once
#include <cstddef>

#include "device_pool.h"

namespace born {

// While it lives this thread's allocations and waits are allowed beside a capture of another thread.
struct LeavesCapturesAlone {
    hipStreamCaptureMode mode = hipStreamCaptureModeRelaxed;
    const bool relaxed = hipThreadExchangeStreamCaptureMode(&mode) == hipSuccess;
    ~LeavesCapturesAlone() {
        if (relaxed) (void)hipThreadExchangeStreamCaptureMode(&mode);
    }
};

// bytes of device memory for *p.  Under capture nothing happens (the next call may ask again); where there is no memory *refused says so
// and no call asks again.
inline void take_once(hipStream_t st, size_t bytes, void **p, bool *refused) {
    if (*p || *refused) return;
    hipStreamCaptureStatus capturing = hipStreamCaptureStatusNone;
    if (st && hipStreamIsCapturing(st, &capturing) != hipSuccess) {
        (void)hipGetLastError();
        return;
    }
    if (capturing != hipStreamCaptureStatusNone) return;
    const LeavesCapturesAlone relaxed;
    if (device_malloc(p, bytes) == hipSuccess) return;
    (void)hipGetLastError();
    *p = nullptr;
    *refused = true;
}

}  // namespace born
