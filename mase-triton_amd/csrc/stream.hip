// What callers ask about streams and events beside the kernels.
#include "../../include/mase_hip_linear.h"
#include "mase_host.h"

// (in the usual mode of a thread a query ends whatever capture is under way; relaxed, it concerns the event alone)
extern "C" int mase_hip_event_done(void* event) {
    if (!event) return 0;
    hipStreamCaptureMode mode = hipStreamCaptureModeRelaxed;
    if (hipThreadExchangeStreamCaptureMode(&mode) != hipSuccess) return (void)hipGetLastError(), 0;
    const hipError_t e = hipEventQuery(static_cast<hipEvent_t>(event));
    if (e != hipSuccess) (void)hipGetLastError();      // (not ready: not for the next launch to report)
    if (hipThreadExchangeStreamCaptureMode(&mode) != hipSuccess) (void)hipGetLastError();
    return e == hipSuccess;
}
