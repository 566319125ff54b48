// The context's scratch block (see aq_workspace.h).  Host code only.
#include "aq_workspace.h"

#include "../../include/aq_mi355.h"

namespace aq {

namespace {

bool capturing(hipStream_t stream) {
    hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;
    return stream != nullptr && hipStreamIsCapturing(stream, &cs) == hipSuccess && cs != hipStreamCaptureStatusNone;
}

size_t with_headroom(size_t need) { return need + need / 4; }  // prompts grow a little from call to call

}  // namespace

hipError_t workspace_open(Workspace* ws, size_t bytes) {
    const hipError_t rc = hipEventCreateWithFlags(&ws->left, hipEventDisableTiming);
    if (rc != hipSuccess || bytes == 0) return rc;
    if (const hipError_t none = hipMalloc(&ws->ptr, bytes)) return none;
    ws->bytes = bytes;
    return hipSuccess;
}

void workspace_close(Workspace* ws) {
    if (ws->ptr) (void)hipFree(ws->ptr);
    ws->ptr = nullptr;
    ws->bytes = 0;
    if (ws->left) (void)hipEventDestroy(ws->left);
    ws->left = nullptr;
}

hipError_t workspace_use(hipStream_t stream, Workspace* ws) {
    if (ws->left_pending && !capturing(stream)) {  // (recorded work runs at a replay, which comes through here itself)
        const hipError_t rc = hipStreamWaitEvent(stream, ws->left, 0);
        if (rc != hipSuccess) return rc;
        ws->left_pending = false;
    }
    ws->used = ws->touched = true;
    return hipSuccess;
}

hipError_t workspace_leave(hipStream_t stream, Workspace* ws) {
    if (!ws->used) return hipSuccess;
    ws->used = false;
    if (capturing(stream)) return hipSuccess;  // what ran before the capture was noted when it began
    hipError_t rc = hipEventRecord(ws->left, stream);
    if (rc == hipSuccess) {
        ws->left_pending = true;
        return rc;
    }
    // the caller has destroyed the stream already: what it still runs is waited for here
    (void)hipGetLastError();
    return hipDeviceSynchronize();
}

bool workspace_may_grow(const Workspace* ws, size_t need, hipStream_t stream) { return ws->bytes >= need || !capturing(stream); }

int workspace_reserve(hipStream_t stream, Workspace* ws, size_t need, FailFn fail) {
    hipError_t rc = workspace_use(stream, ws);
    if (rc != hipSuccess) return fail((int)rc, "rocm.hip.hipStreamWaitEvent: HIP returned %d", (int)rc);
    if (ws->bytes >= need) return AQ_OK;
    if (capturing(stream))
        return fail(AQ_ERR_UNSUPPORTED,
                    "the context's workspace must grow to %zu bytes, which cannot happen during stream capture; "
                    "run the call once, or call aq_reserve_workspace / aq_reserve_workspace_bytes, before capturing", need);
    rc = hipStreamSynchronize(stream);
    if (rc != hipSuccess) return fail((int)rc, "rocm.hip.hipStreamSynchronize: HIP returned %d", (int)rc);
    if (ws->ptr) (void)hipFree(ws->ptr);
    ws->ptr = nullptr;
    ws->bytes = 0;
    ws->generation++;  // graphs captured over the old block must not run again
    rc = hipMalloc(&ws->ptr, with_headroom(need));
    if (rc != hipSuccess) return fail(AQ_ERR_NOMEM, "aq_qmm: cannot allocate a %zu-byte workspace (HIP %d)", with_headroom(need), (int)rc);
    ws->bytes = with_headroom(need);
    return AQ_OK;
}

}  // namespace aq
