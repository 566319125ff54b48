// Scratch memory a context lends to its calls: one device block, grown on demand, never while a capture is open.
//
// Its users follow each other on the context's stream.  When the context moves to another stream, the work that the old
// one still holds over the block is kept in order by an event: recorded when the stream is left (workspace_leave), waited for
// by the first use on the new one.
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
// The context goes from `stream` to another one, or begins a capture on it.
hipError_t workspace_leave(hipStream_t stream, Workspace* ws);

}  // namespace aq
