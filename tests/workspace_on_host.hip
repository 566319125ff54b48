// The context's scratch block (csrc/aq_workspace.hip) against a HIP runtime of its own: the entry points it calls are defined
// here and write down what they were asked, so that order, growth and refusals can be checked without a GPU.
#include "aq_workspace.h"

#include "../include/aq_mi355.h"

#include <cstdarg>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <string>
#include <vector>

static std::vector<std::string> calls;  // in order
static int live_blocks = 0, next_id = 1, record_fails = 0;
static size_t memory = 1 << 20;  // bytes hipMalloc may still hand out
static hipStream_t capturing_stream = nullptr, destroyed_stream = nullptr;
static void must_exist(hipStream_t s) {  // the runtime reads the object behind a handle without a look whether it is there
    if (s && s == destroyed_stream) {
        puts("a destroyed stream was asked for");
        exit(1);
    }
}

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
    must_exist(s);
    if (record_fails) return hipErrorUnknown;
    note("record %s", name(s).c_str());
    return hipSuccess;
}
hipError_t hipStreamWaitEvent(hipStream_t s, hipEvent_t, unsigned) {
    must_exist(s);
    note("wait %s", name(s).c_str());
    return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t s) {
    must_exist(s);
    note("sync %s", name(s).c_str());
    return hipSuccess;
}
hipError_t hipDeviceSynchronize(void) {
    note("sync device");
    return hipSuccess;
}
hipError_t hipStreamIsCapturing(hipStream_t s, hipStreamCaptureStatus* cs) {
    must_exist(s);
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

static hipError_t note_and_leave(hipStream_t stream, aq::Workspace* ws) {
    const hipError_t rc = aq::workspace_note(stream, ws), left = aq::workspace_leave(ws);
    return rc != hipSuccess ? rc : left;
}

static void use_on_another_stream_waits_for_the_last_one() {
    aq::Workspace ws;
    EXPECT(aq::workspace_open(&ws, 0) == hipSuccess);
    EXPECT(aq::workspace_reserve(A, &ws, 400, quiet) == 0 && ws.bytes == 500);
    EXPECT(seen({"sync A", "malloc 500"}));
    EXPECT(note_and_leave(A, &ws) == hipSuccess && seen({"record A"}));
    EXPECT(aq::workspace_reserve(B, &ws, 100, quiet) == 0 && seen({"wait B"}));  // before any kernel of the call
    EXPECT(aq::workspace_reserve(B, &ws, 100, quiet) == 0 && seen({}));          // once
    EXPECT(note_and_leave(B, &ws) == hipSuccess && seen({"record B"}));
    // a stream that never used the block is passed through: the one behind it still waits
    EXPECT(note_and_leave(A, &ws) == hipSuccess && seen({}));
    EXPECT(aq::workspace_use(C, &ws) == hipSuccess && seen({"wait C"}));
    // growth frees the block behind everybody's work
    EXPECT(note_and_leave(C, &ws) == hipSuccess && seen({"record C"}));
    EXPECT(aq::workspace_reserve(A, &ws, 800, quiet) == 0 && seen({"wait A", "sync A", "free", "malloc 1000"}));
    // no event to be had: the stream is waited for instead
    record_fails = 1;
    EXPECT(note_and_leave(A, &ws) == hipSuccess && seen({"sync A"}));
    record_fails = 0;
    aq::workspace_close(&ws);
    calls.clear();
    EXPECT(live_blocks == 0);
}

static void a_stream_may_be_destroyed_before_it_is_left() {
    aq::Workspace ws;
    EXPECT(aq::workspace_open(&ws, 1000) == hipSuccess && seen({"malloc 1000"}));
    EXPECT(aq::workspace_use(A, &ws) == hipSuccess && aq::workspace_note(A, &ws) == hipSuccess && seen({"record A"}));  // a call
    EXPECT(aq::workspace_note(A, &ws) == hipSuccess && seen({}));
    destroyed_stream = A;
    EXPECT(aq::workspace_leave(&ws) == hipSuccess && seen({}));
    EXPECT(aq::workspace_use(B, &ws) == hipSuccess && seen({"wait B"}));
    // uses that were not noted, captured ones aside: the device is waited for, once
    EXPECT(aq::workspace_note(B, &ws, false) == hipSuccess && seen({}));
    destroyed_stream = B;
    EXPECT(aq::workspace_leave(&ws) == hipSuccess && seen({"sync device"}));
    EXPECT(aq::workspace_leave(&ws) == hipSuccess && aq::workspace_use(C, &ws) == hipSuccess && seen({}));
    capturing_stream = C;
    EXPECT(aq::workspace_note(C, &ws, false) == hipSuccess && aq::workspace_leave(&ws) == hipSuccess && seen({}));
    capturing_stream = destroyed_stream = nullptr;
    aq::workspace_close(&ws);
    calls.clear();
}

static void captured_uses_wait_for_nothing_and_are_ordered_when_replayed() {
    aq::Workspace ws;
    EXPECT(aq::workspace_open(&ws, 1000) == hipSuccess && seen({"malloc 1000"}));
    EXPECT(aq::workspace_use(A, &ws) == hipSuccess);
    EXPECT(note_and_leave(A, &ws) == hipSuccess && seen({"record A"}));
    capturing_stream = B;
    EXPECT(aq::workspace_reserve(B, &ws, 600, quiet) == 0 && aq::workspace_note(B, &ws) == hipSuccess && seen({}));  // recorded, not run
    EXPECT(aq::workspace_reserve(B, &ws, 2000, quiet) != 0 && seen({}) && ws.bytes == 1000);
    capturing_stream = nullptr;
    EXPECT(aq::workspace_use(B, &ws) == hipSuccess && seen({"wait B"}));  // the replay
    // a capture begins on the stream in use, and the context leaves it while it is open
    EXPECT(note_and_leave(B, &ws) == hipSuccess && seen({"record B"}));
    capturing_stream = B;
    EXPECT(aq::workspace_use(B, &ws) == hipSuccess && note_and_leave(B, &ws) == hipSuccess && seen({}));
    EXPECT(aq::workspace_use(C, &ws) == hipSuccess && seen({"wait C"}));
    capturing_stream = nullptr;
    aq::workspace_close(&ws);
    calls.clear();
    EXPECT(live_blocks == 0);
}

static void an_offer_that_cannot_be_met_changes_nothing() {
    aq::Workspace ws;
    EXPECT(aq::workspace_open(&ws, 0) == hipSuccess);
    EXPECT(aq::workspace_reserve(A, &ws, 400, quiet) == 0 && seen({"sync A", "malloc 500"}));
    const void* const before = ws.ptr;
    const uint64_t generation = ws.generation, moves = ws.moves;
    capturing_stream = A;
    EXPECT(!aq::workspace_offer(A, &ws, 501) && aq::workspace_offer(A, &ws, 500) && seen({}));
    capturing_stream = nullptr;
    const size_t all = memory;
    memory = 700;
    EXPECT(!aq::workspace_offer(A, &ws, 701) && seen({}));
    EXPECT(ws.ptr == before && ws.bytes == 500 && ws.moves == moves && ws.generation == generation);
    EXPECT(aq::workspace_offer(A, &ws, 700) && ws.bytes == 700);  // no room for more than the call needs
    EXPECT(seen({"malloc 700", "sync A", "free"}));
    EXPECT(ws.moves != moves && ws.generation == generation);
    memory = all;
    EXPECT(aq::workspace_reserve(A, &ws, 701, quiet) == 0 && ws.generation == generation + 1);
    memory = 0;
    EXPECT(aq::workspace_reserve(A, &ws, 5000, quiet) == AQ_ERR_NOMEM && ws.bytes == 0 && ws.ptr == nullptr);
    memory = all;
    EXPECT(aq::workspace_reserve(A, &ws, 100, quiet) == 0 && ws.bytes == 125);
    aq::workspace_close(&ws);
    calls.clear();
    EXPECT(live_blocks == 0);
}

static void a_block_that_a_graph_keeps_outlives_growth() {
    aq::Workspace ws;
    EXPECT(aq::workspace_open(&ws, 1000) == hipSuccess);
    ws.touched = ws.required = false;  // a capture begins
    capturing_stream = A;
    EXPECT(aq::workspace_offer(A, &ws, 900) && ws.touched && !ws.required);
    capturing_stream = nullptr;
    std::shared_ptr<aq::WorkspaceBlock> kept = ws.block;
    EXPECT(aq::workspace_offer(A, &ws, 2000) && live_blocks == 2 && ws.ptr != kept->ptr);
    EXPECT(aq::workspace_reserve(A, &ws, 4000, quiet) == 0 && live_blocks == 2 && ws.required);
    kept.reset();  // the graph is destroyed
    EXPECT(live_blocks == 1);
    aq::workspace_close(&ws);
    calls.clear();
    EXPECT(live_blocks == 0);
}

int main() {
    an_offer_that_cannot_be_met_changes_nothing();
    a_block_that_a_graph_keeps_outlives_growth();
    use_on_another_stream_waits_for_the_last_one();
    a_stream_may_be_destroyed_before_it_is_left();
    captured_uses_wait_for_nothing_and_are_ordered_when_replayed();
    puts("ok");
    return 0;
}
