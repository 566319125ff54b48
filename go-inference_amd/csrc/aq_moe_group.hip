// Routes grouped by expert, on the device: what lets a gathered projection of many routes (a prompt, a decode batch larger
// than the expert count) read every expert's weights once instead of once per route.
//
// Stands in for the host grouping of the reference's batch path (hipGemma4MoEBatchRouteGroups,
// go/engine/hip/hip_gemma4_moe.go:294-366), whose ids come back to the host first.  Here the expert ids stay where the
// router wrote them: one workgroup counts the routes of every expert, places them side by side and cuts every expert's run
// into chunks that one workgroup tile of the matmul (or token-tile) kernels takes as its rows of x.  The list has as many
// entries as the ids ask for; the launches behind it are sized for the most there can be and read the count here.
//
// Bound: latency, and the scattered places.  Two passes over 4 bytes a route with LDS counters and one scan over the experts, one
// workgroup because the passes depend on each other through the counters (a grid-wide meeting costs more).  4096 routes over 128
// experts in a kernel trace: places stored to memory one by one, loads each behind a branch 11.7 us -> 7.9; 876 routes over 32 4.9 -> 5.1.
#include "aq_moe_group.h"

namespace aq {

template <bool STAGED>
__global__ __launch_bounds__(kGroupThreads) void moe_group_kernel(const RouteGroupArgs a) {
    extern __shared__ __attribute__((aligned(16))) int32_t counter[];
    group_routes<STAGED>(a, counter);
}

hipError_t moe_group_launch(const RouteGroupArgs& a, hipStream_t stream) {
    const size_t counters = group_counter_bytes(a), staged = group_staged_bytes(a);
    if (staged > 128 * 1024) {
        hipLaunchKernelGGL(moe_group_kernel<false>, dim3(1), dim3(kGroupThreads), counters, stream, a);
    } else {
        if (hipError_t rc = ensure_dynamic_lds(reinterpret_cast<const void*>(moe_group_kernel<true>), staged)) return rc;
        hipLaunchKernelGGL(moe_group_kernel<true>, dim3(1), dim3(kGroupThreads), staged, stream, a);
    }
    return hipGetLastError();
}

}  // namespace aq
