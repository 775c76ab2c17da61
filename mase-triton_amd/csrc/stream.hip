// What callers ask about streams and events beside the kernels.
#include "../../include/mase_hip_linear.h"
#include "mase_host.h"

// Asked in the mode in which a query concerns its own event or stream alone (in the usual mode of a thread it ends whatever capture is under way), and not at
// all of a captured stream, whose capture a query of it or of its earlier events ends in any mode.
extern "C" int mase_hip_stream_done(void* stream, void* event) {
    hipStreamCaptureMode mode = hipStreamCaptureModeRelaxed;
    if (hipThreadExchangeStreamCaptureMode(&mode) != hipSuccess) return (void)hipGetLastError(), 0;
    hipStreamCaptureStatus status = hipStreamCaptureStatusNone;
    hipError_t e = hipStreamIsCapturing(static_cast<hipStream_t>(stream), &status);
    if (e == hipSuccess)
        e = status != hipStreamCaptureStatusNone ? hipErrorNotReady : event ? hipEventQuery(static_cast<hipEvent_t>(event)) : hipStreamQuery(static_cast<hipStream_t>(stream));
    if (e != hipSuccess) (void)hipGetLastError();      // (not ready: not for the next launch to report)
    if (hipThreadExchangeStreamCaptureMode(&mode) != hipSuccess) (void)hipGetLastError();
    return e == hipSuccess;
}
