// Routes grouped by expert, on the device: what lets a gathered projection of many routes (a prompt, a decode batch larger
// than the expert count) read every expert's weights once instead of once per route.
//
// Stands in for the host grouping of the reference's batch path (hipGemma4MoEBatchRouteGroups,
// go/engine/hip/hip_gemma4_moe.go:294-366), whose ids come back to the host first.  Here the expert ids stay where the
// router wrote them: one workgroup counts the routes of every expert, places them side by side and cuts every expert's run
// into chunks that one workgroup tile of the matmul (or token-tile) kernels takes as its rows of x.  The list has as many
// entries as the ids ask for; the launches behind it are sized for the most there can be and read the count here.
//
// Bound: latency.  Two passes over 4 bytes a route with LDS counters and one scan over the experts, one workgroup because
// the passes depend on each other through the counters (4096 routes over 128 experts: 11 us in a kernel trace; a grid-wide
// meeting costs more than that).
#include "aq_device.h"
#include "aq_kernels.h"

namespace aq {

constexpr int kGroupThreads = 1024;

__global__ __launch_bounds__(kGroupThreads) void moe_group_kernel(const RouteGroupArgs a) {
    extern __shared__ int32_t counter[];  // [num_experts] routes of the expert, then the next free place of its run
    __shared__ int32_t wave_rows[kGroupThreads / kWave], wave_chunks[kGroupThreads / kWave];
    const int tid = threadIdx.x, lane = tid & (kWave - 1), wave = tid >> 6;
    const int E = a.num_experts;
    for (int e = tid; e < E; e += kGroupThreads) counter[e] = 0;
    __syncthreads();

    // expert of a route; a route whose ids are out of range goes with expert 0 (bit 30 set), its outputs become zeros
    constexpr int kBad = 1 << 30;
    auto expert_of = [&](int r) {
        const int e = a.rhs[r], x = a.lhs ? a.lhs[r] : 0;
        return e < 0 || e >= E || x < 0 || x >= a.x_rows ? kBad : e;
    };
    constexpr int HOLD = 8;  // up to 8192 routes: the ids are read once and kept
    int held[HOLD];
#pragma unroll
    for (int i = 0; i < HOLD; i++) {
        const int r = tid + i * kGroupThreads;
        held[i] = r < a.routes ? expert_of(r) : -1;
    }
#pragma unroll
    for (int i = 0; i < HOLD; i++)
        if (held[i] >= 0) atomicAdd(&counter[held[i] & (kBad - 1)], 1);
    for (int r = tid + HOLD * kGroupThreads; r < a.routes; r += kGroupThreads) atomicAdd(&counter[expert_of(r) & (kBad - 1)], 1);
    __syncthreads();

    // exclusive sums over the experts of (padded rows, chunks); thread t takes experts t * per .. t * per + per - 1
    const int per = (E + kGroupThreads - 1) / kGroupThreads;
    const int e0 = min(tid * per, E), e1 = min(e0 + per, E);
    auto padded = [&](int n) { return (n + a.pad - 1) / a.pad * a.pad; };
    int rows = 0, chunks = 0;
    for (int e = e0; e < e1; e++) {
        rows += padded(counter[e]);
        chunks += (counter[e] + a.chunk_rows - 1) / a.chunk_rows;
    }
    int rows_to = rows, chunks_to = chunks;  // inclusive inside the wavefront
#pragma unroll
    for (int o = 1; o < kWave; o <<= 1) {
        const int r = __shfl_up(rows_to, o, kWave), c = __shfl_up(chunks_to, o, kWave);
        if (lane >= o) rows_to += r, chunks_to += c;
    }
    if (lane == kWave - 1) wave_rows[wave] = rows_to, wave_chunks[wave] = chunks_to;
    __syncthreads();
    int row = rows_to - rows, chunk = chunks_to - chunks, all_rows = 0, all_chunks = 0;
    for (int w = 0; w < kGroupThreads / kWave; w++) {
        if (w < wave) row += wave_rows[w], chunk += wave_chunks[w];
        all_rows += wave_rows[w];
        all_chunks += wave_chunks[w];
    }
    for (int e = e0; e < e1; e++) {
        const int n = counter[e], end = row + padded(n);
        for (int c = 0; c < n; c += a.chunk_rows) a.chunks[chunk++] = RouteChunk{e, row + c, min(a.chunk_rows, n - c), 0};
        for (int i = row + n; i < end; i++) a.route_x[i] = -1, a.route_of[i] = -1;
        counter[e] = row;
        row = end;
    }
    for (int c = all_chunks + tid; c < a.most_chunks; c += kGroupThreads) a.chunks[c] = RouteChunk{0, 0, 0, 0};
    if (tid == 0) *a.nchunks = all_chunks, *a.live_rows = all_rows;
    __syncthreads();

    auto place = [&](int r, int e) {
        const int at = atomicAdd(&counter[e & (kBad - 1)], 1);
        const bool bad = (e & kBad) != 0;
        a.route_x[at] = bad ? -1 : a.lhs ? a.lhs[r] : 0;
        a.route_of[at] = bad ? r | INT32_MIN : r;
    };
#pragma unroll
    for (int i = 0; i < HOLD; i++)
        if (held[i] >= 0) place(tid + i * kGroupThreads, held[i]);
    for (int r = tid + HOLD * kGroupThreads; r < a.routes; r += kGroupThreads) place(r, expert_of(r));
}

hipError_t moe_group_launch(const RouteGroupArgs& a, hipStream_t stream) {
    hipLaunchKernelGGL(moe_group_kernel, dim3(1), dim3(kGroupThreads), (size_t)a.num_experts * 4, stream, a);
    return hipGetLastError();
}

}  // namespace aq
