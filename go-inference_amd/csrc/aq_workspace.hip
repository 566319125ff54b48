// The context's scratch block (see aq_workspace.h).  Host code only.
#include "aq_workspace.h"

#include <new>

#include "../../include/aq_mi355.h"

namespace aq {

namespace {

bool capturing(hipStream_t stream) {
    hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;
    return stream != nullptr && hipStreamIsCapturing(stream, &cs) == hipSuccess && cs != hipStreamCaptureStatusNone;
}

hipError_t allocate(size_t bytes, std::shared_ptr<WorkspaceBlock>* out) {
    std::shared_ptr<WorkspaceBlock> b;
    try {
        b = std::make_shared<WorkspaceBlock>();
    } catch (const std::bad_alloc&) {
        return hipErrorOutOfMemory;
    }
    const hipError_t rc = hipMalloc(&b->ptr, bytes);
    if (rc != hipSuccess) {
        b->ptr = nullptr;
        (void)hipGetLastError();  // the caller has another way, or reports it itself
        return rc;
    }
    b->bytes = bytes;
    *out = std::move(b);
    return hipSuccess;
}

void put(Workspace* ws, std::shared_ptr<WorkspaceBlock> b) {
    ws->block = std::move(b);
    ws->ptr = ws->block ? ws->block->ptr : nullptr;
    ws->bytes = ws->block ? ws->block->bytes : 0;
    ws->moves++;
}

size_t with_headroom(size_t need) { return need + need / 4; }  // prompts grow a little from call to call

}  // namespace

WorkspaceBlock::~WorkspaceBlock() {
    if (ptr) (void)hipFree(ptr);
}

hipError_t workspace_open(Workspace* ws, size_t bytes) {
    const hipError_t rc = hipEventCreateWithFlags(&ws->left, hipEventDisableTiming);
    if (rc != hipSuccess || bytes == 0) return rc;
    std::shared_ptr<WorkspaceBlock> b;
    if (const hipError_t none = allocate(bytes, &b)) return none;
    put(ws, std::move(b));
    return hipSuccess;
}

void workspace_close(Workspace* ws) {
    put(ws, nullptr);
    if (ws->left) (void)hipEventDestroy(ws->left);
    ws->left = nullptr;
}

hipError_t workspace_use(hipStream_t stream, Workspace* ws) {
    if (ws->left_pending && !capturing(stream)) {  // (recorded work runs at a replay, which comes through here itself)
        const hipError_t rc = hipStreamWaitEvent(stream, ws->left, 0);
        if (rc != hipSuccess) return rc;
        ws->left_pending = false;
    }
    ws->used = ws->unnoted = ws->touched = true;
    return hipSuccess;
}

hipError_t workspace_note(hipStream_t stream, Workspace* ws, bool record) {
    if (!ws->unnoted) return hipSuccess;
    if (capturing(stream)) {  // recorded, not run; what ran before the capture was noted when it began
        ws->unnoted = false;
        return hipSuccess;
    }
    if (!record) return hipSuccess;
    ws->unnoted = false;
    hipError_t rc = hipEventRecord(ws->left, stream);
    if (rc != hipSuccess) {
        (void)hipGetLastError();
        rc = hipStreamSynchronize(stream);  // nothing is left to wait for
    }
    return rc;
}

hipError_t workspace_leave(Workspace* ws) {
    if (!ws->used) return hipSuccess;
    ws->used = false;
    if (!ws->unnoted) {
        ws->left_pending = true;
        return hipSuccess;
    }
    ws->unnoted = ws->left_pending = false;
    return hipDeviceSynchronize();
}

bool workspace_may_grow(const Workspace* ws, size_t need, hipStream_t stream) { return ws->bytes >= need || !capturing(stream); }

int workspace_reserve(hipStream_t stream, Workspace* ws, size_t need, FailFn fail) {
    ws->required = true;
    hipError_t rc = workspace_use(stream, ws);
    if (rc != hipSuccess) return fail((int)rc, "rocm.hip.hipStreamWaitEvent: HIP returned %d", (int)rc);
    if (ws->bytes >= need) return AQ_OK;
    if (capturing(stream))
        return fail(AQ_ERR_UNSUPPORTED,
                    "the context's workspace must grow to %zu bytes, which cannot happen during stream capture; "
                    "run the call once, or call aq_reserve_workspace / aq_reserve_workspace_bytes, before capturing", need);
    rc = hipStreamSynchronize(stream);
    if (rc != hipSuccess) return fail((int)rc, "rocm.hip.hipStreamSynchronize: HIP returned %d", (int)rc);
    put(ws, nullptr);
    ws->generation++;  // graphs that need the old block must not run again
    std::shared_ptr<WorkspaceBlock> b;
    rc = allocate(with_headroom(need), &b);
    if (rc != hipSuccess) return fail(AQ_ERR_NOMEM, "aq_qmm: cannot allocate a %zu-byte workspace (HIP %d)", with_headroom(need), (int)rc);
    put(ws, std::move(b));
    return AQ_OK;
}

bool workspace_offer(hipStream_t stream, Workspace* ws, size_t need) {
    std::shared_ptr<WorkspaceBlock> b;
    if (ws->bytes < need) {
        if (capturing(stream)) return false;
        if (allocate(with_headroom(need), &b) != hipSuccess && allocate(need, &b) != hipSuccess) return false;
    }
    if (workspace_use(stream, ws) != hipSuccess) return false;
    if (b) {
        // (the old block may be the last reference's to free: its users are done first)
        if (ws->block && hipStreamSynchronize(stream) != hipSuccess) return false;
        put(ws, std::move(b));
    }
    return true;
}

}  // namespace aq
