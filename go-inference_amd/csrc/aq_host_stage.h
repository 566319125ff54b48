// How the entry points that take host slices bring them to the device (aq_matvec_host, aq_proj_quant_matmul_host): one
// staged upload per call instead of an allocation, a synchronous copy from pageable memory and a free per array.
#pragma once
#include <hip/hip_runtime.h>
#include <stddef.h>
#include <stdint.h>

namespace aq {

// One host array of an upload: `bytes` device bytes at offset `at` (a multiple of 256) of the device block.
// from_f32: src holds fp32 values, which arrive as bf16 (round to nearest even; NaN quiet).
struct HostPart {
    const void* src;
    size_t bytes, at;
    bool from_f32;
};

class HostStage {
public:
    ~HostStage();
    // Makes the device block hold at least `bytes` (before an upload whose call wants room behind the parts).
    hipError_t reserve_device(size_t bytes) { return grow(&dev_, &dev_bytes_, bytes, false); }
    // Queues the parts' upload on `stream`; *dev is the device block of `total` bytes (a multiple of 256).  The host slices
    // have been read when it returns.
    hipError_t upload(const HostPart* parts, int count, size_t total, hipStream_t stream, char** dev);
    // Pinned host memory of at least `bytes` (at most kMostResults) that kernels may write, for results.
    static constexpr size_t kMostResults = (size_t)16 << 20;
    hipError_t results(size_t bytes, void** host);
    // out[i] = fp32 of n bf16 values, shared out over the worker threads when there are many.
    void widen(float* out, const uint16_t* in, size_t n);
    // Ends a call (the stream has been waited for): a device block larger than what is kept between calls is freed.
    void finish();
    // Device memory kept between calls.
    size_t device_bytes() const { return dev_bytes_; }

private:
    struct Pool;
    Pool* pool_ = nullptr;
    char* pinned_ = nullptr;  // ring of pieces
    char* dev_ = nullptr;
    void* out_ = nullptr;
    size_t pinned_bytes_ = 0, dev_bytes_ = 0, out_bytes_ = 0;
    hipEvent_t event_ = nullptr;  // created when an upload is longer than the ring
    hipError_t grow(char** p, size_t* have, size_t want, bool host);
};

}  // namespace aq
