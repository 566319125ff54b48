// The context's scratch block (csrc/aq_workspace.hip) against a HIP runtime of its own: the entry points it calls are defined
// here and write down what they were asked, so that order, growth and refusals can be checked without a GPU.
#include "aq_workspace.h"

#include <cstdarg>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <string>
#include <vector>

static std::vector<std::string> calls;  // in order
static int live_blocks = 0, next_id = 1, record_fails = 0;
static size_t memory = 1 << 20;  // bytes hipMalloc may still hand out
static hipStream_t capturing_stream = nullptr;

static void note(const char* fmt, ...) {
    char b[128];
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(b, sizeof b, fmt, ap);
    va_end(ap);
    calls.push_back(b);
}
static std::string name(hipStream_t s) { return s ? std::string(1, (char)reinterpret_cast<uintptr_t>(s)) : "0"; }

extern "C" {
hipError_t hipMalloc(void** p, size_t n) {
    if (n > memory) return hipErrorOutOfMemory;
    memory -= n;
    size_t* b = static_cast<size_t*>(malloc(sizeof(size_t)));
    *b = n;
    *p = b;
    live_blocks++;
    note("malloc %zu", n);
    return hipSuccess;
}
hipError_t hipFree(void* p) {
    memory += *static_cast<size_t*>(p);
    free(p);
    live_blocks--;
    note("free");
    return hipSuccess;
}
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) {
    *e = reinterpret_cast<hipEvent_t>((uintptr_t)next_id++);
    return hipSuccess;
}
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t s) {
    if (record_fails) return hipErrorContextIsDestroyed;
    note("record %s", name(s).c_str());
    return hipSuccess;
}
hipError_t hipStreamWaitEvent(hipStream_t s, hipEvent_t, unsigned) {
    note("wait %s", name(s).c_str());
    return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t s) {
    note("sync %s", name(s).c_str());
    return hipSuccess;
}
hipError_t hipDeviceSynchronize(void) {
    note("sync device");
    return hipSuccess;
}
hipError_t hipStreamIsCapturing(hipStream_t s, hipStreamCaptureStatus* cs) {
    *cs = s == capturing_stream && s ? hipStreamCaptureStatusActive : hipStreamCaptureStatusNone;
    return hipSuccess;
}
hipError_t hipGetLastError(void) { return hipSuccess; }
}

static int quiet(int code, const char*, ...) { return code; }

#define EXPECT(cond)                                                                \
    do {                                                                            \
        if (!(cond)) {                                                              \
            printf("%s:%d: %s\n", __func__, __LINE__, #cond);                       \
            for (auto& c : calls) printf("    %s\n", c.c_str());                    \
            exit(1);                                                                \
        }                                                                           \
    } while (0)

static bool seen(std::vector<std::string> want) {
    const bool same = calls == want;
    if (same) calls.clear();
    return same;
}

static const hipStream_t A = reinterpret_cast<hipStream_t>((uintptr_t)'A'), B = reinterpret_cast<hipStream_t>((uintptr_t)'B'),
                         C = reinterpret_cast<hipStream_t>((uintptr_t)'C');

static void use_on_another_stream_waits_for_the_last_one() {
    aq::Workspace ws;
    EXPECT(aq::workspace_open(&ws, 0) == hipSuccess);
    EXPECT(aq::workspace_reserve(A, &ws, 400, quiet) == 0 && ws.bytes == 500);
    EXPECT(seen({"sync A", "malloc 500"}));
    EXPECT(aq::workspace_leave(A, &ws) == hipSuccess && seen({"record A"}));
    EXPECT(aq::workspace_reserve(B, &ws, 100, quiet) == 0 && seen({"wait B"}));  // before any kernel of the call
    EXPECT(aq::workspace_reserve(B, &ws, 100, quiet) == 0 && seen({}));          // once
    EXPECT(aq::workspace_leave(B, &ws) == hipSuccess && seen({"record B"}));
    // a stream that never used the block is passed through: the one behind it still waits
    EXPECT(aq::workspace_leave(A, &ws) == hipSuccess && seen({}));
    EXPECT(aq::workspace_use(C, &ws) == hipSuccess && seen({"wait C"}));
    // growth frees the block behind everybody's work
    EXPECT(aq::workspace_leave(C, &ws) == hipSuccess && seen({"record C"}));
    EXPECT(aq::workspace_reserve(A, &ws, 800, quiet) == 0 && seen({"wait A", "sync A", "free", "malloc 1000"}));
    // a stream that is gone when it is left: the device is waited for instead
    record_fails = 1;
    EXPECT(aq::workspace_leave(A, &ws) == hipSuccess && seen({"sync device"}));
    record_fails = 0;
    EXPECT(aq::workspace_use(B, &ws) == hipSuccess && seen({}));
    aq::workspace_close(&ws);
    calls.clear();
    EXPECT(live_blocks == 0);
}

static void captured_uses_wait_for_nothing_and_are_ordered_when_replayed() {
    aq::Workspace ws;
    EXPECT(aq::workspace_open(&ws, 1000) == hipSuccess && seen({"malloc 1000"}));
    EXPECT(aq::workspace_use(A, &ws) == hipSuccess);
    EXPECT(aq::workspace_leave(A, &ws) == hipSuccess && seen({"record A"}));
    capturing_stream = B;
    EXPECT(aq::workspace_reserve(B, &ws, 600, quiet) == 0 && seen({}));  // recorded, not run
    EXPECT(aq::workspace_reserve(B, &ws, 2000, quiet) != 0 && seen({}) && ws.bytes == 1000);
    capturing_stream = nullptr;
    EXPECT(aq::workspace_use(B, &ws) == hipSuccess && seen({"wait B"}));  // the replay
    // a capture begins on the stream in use, and the context leaves it while it is open
    EXPECT(aq::workspace_leave(B, &ws) == hipSuccess && seen({"record B"}));
    capturing_stream = B;
    EXPECT(aq::workspace_use(B, &ws) == hipSuccess && aq::workspace_leave(B, &ws) == hipSuccess && seen({}));
    EXPECT(aq::workspace_use(C, &ws) == hipSuccess && seen({"wait C"}));
    capturing_stream = nullptr;
    aq::workspace_close(&ws);
    calls.clear();
    EXPECT(live_blocks == 0);
}

int main() {
    use_on_another_stream_waits_for_the_last_one();
    captured_uses_wait_for_nothing_and_are_ordered_when_replayed();
    puts("ok");
    return 0;
}
