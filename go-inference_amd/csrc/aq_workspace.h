// Scratch memory a context lends to its calls: one device block, grown on demand, never while a capture is open.
//
// Its users follow each other on the context's stream.  When the context moves to another stream, the work that the old
// one still holds over the block is kept in order by an event: recorded behind the last use (workspace_note), waited for by the
// first use on the new one.  The context's own stream is noted when it is left.  A caller's stream may have been destroyed by
// then, and the runtime must not be asked for it; noting every use on it as it ends costs 3 us of the stream (a marker; 40 best
// of 262144 13.9 -> 17.0 us), which a program that stays on one stream would pay for nothing.  So the first time that one is
// left the device is waited for, and from then on uses on callers' streams are noted (CallLock in aq_api.hip).
#pragma once
#include <hip/hip_runtime_api.h>
#include <stddef.h>
#include <stdint.h>

#include <memory>

namespace aq {

typedef int (*FailFn)(int code, const char* fmt, ...);

struct WorkspaceBlock {
    void* ptr = nullptr;
    size_t bytes = 0;
    ~WorkspaceBlock();
};

// `generation` counts the growths that gave the old block up (workspace_reserve).  `touched` is set by every use, `required`
// by the uses of calls that have no route without scratch; both are cleared when a capture begins, so that the graph knows
// what it recorded.
struct Workspace {
    std::shared_ptr<WorkspaceBlock> block;  // shared with the graphs recorded over it
    void* ptr = nullptr;                    // of block
    size_t bytes = 0;
    uint64_t generation = 0;
    uint64_t moves = 0;  // every change of block, whoever asked for it
    bool touched = false, required = false;
    hipEvent_t left = nullptr;
    bool used = false;          // work over the block was queued on the current stream since it became current
    bool unnoted = false;       // ... since `left` was recorded
    bool left_pending = false;  // `left` stands for work on another stream that the current one has not waited for
};

// The event and a first block of `bytes` (0: none), on the current device; and their end.
hipError_t workspace_open(Workspace* ws, size_t bytes);
void workspace_close(Workspace* ws);
// Makes ws hold at least `need` bytes and orders the call behind the block's other users.  For calls that cannot do without:
// when the block must grow, the stream is drained and the old block freed first (refused while the stream is being captured).
int workspace_reserve(hipStream_t stream, Workspace* ws, size_t need, FailFn fail);
// The same for calls that have another route: false, and nothing changed, when the bytes cannot be had (the stream is being
// captured, or there is no memory).  A new block is made beside the old one; graphs recorded over that keep it.
bool workspace_offer(hipStream_t stream, Workspace* ws, size_t need);
// Whether ws holds `need` bytes or may be made to (not while the stream is being captured).
bool workspace_may_grow(const Workspace* ws, size_t need, hipStream_t stream);
// Orders a use of a block of ws (the current one or one that a graph keeps) on `stream` behind the earlier ones.
hipError_t workspace_use(hipStream_t stream, Workspace* ws);
// Notes the end of what `stream` (the current one) has been given to do over the block (record: with an event; else only that
// recorded work needs none).
hipError_t workspace_note(hipStream_t stream, Workspace* ws, bool record = true);
// The context goes to another stream, or begins a capture: what was noted is for the next use to wait for, and the device is
// waited for here if something was not.
hipError_t workspace_leave(Workspace* ws);

}  // namespace aq
