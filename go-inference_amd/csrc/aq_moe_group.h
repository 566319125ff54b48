// The grouping of routes by expert (aq_moe_group.hip) as one workgroup's work, for launches that do something beside it.
#pragma once
#include "aq_device.h"
#include "aq_kernels.h"

namespace aq {

constexpr int kGroupThreads = 1024;

// STAGED: the two lists of places are put together in LDS and leave it in whole lines.  Places lie all over a list, and a store
// instruction takes about four clocks per line that it touches: 8192 of them were most of this kernel's 11.5 us.
// counter: LDS, [num_experts] routes of the expert, then the next free place of its run; STAGED: behind it the lists.
template <bool STAGED>
__device__ __forceinline__ void group_routes(const RouteGroupArgs& a, int32_t* counter) {
    int32_t* const list_x = STAGED ? counter + (a.num_experts + 3) / 4 * 4 : a.route_x;
    int32_t* const list_of = STAGED ? list_x + (a.most_rows + 3) / 4 * 4 : a.route_of;
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
    int held[HOLD], from[HOLD];
    // (loads without a branch of the lanes around each, or every one of them is waited for before the next is asked for)
#pragma unroll
    for (int i = 0; i < HOLD; i++) held[i] = -1, from[i] = 0;
#pragma unroll
    for (int i = 0; i < HOLD; i++) {
        if (i * kGroupThreads >= a.routes) break;
        const int r = min(tid + i * kGroupThreads, a.routes - 1);
        held[i] = a.rhs[r];
        if (a.lhs) from[i] = a.lhs[r];
    }
#pragma unroll
    for (int i = 0; i < HOLD; i++) {
        if (held[i] < 0 || held[i] >= E || from[i] < 0 || from[i] >= a.x_rows) held[i] = kBad;
        if (tid + i * kGroupThreads >= a.routes) held[i] = -1;
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
#pragma unroll
    for (int w = 0; w < kGroupThreads / kWave; w++) {
        if (w < wave) row += wave_rows[w], chunk += wave_chunks[w];
        all_rows += wave_rows[w];
        all_chunks += wave_chunks[w];
    }
    for (int e = e0; e < e1; e++) {
        const int n = counter[e], end = row + padded(n);
        for (int c = 0; c < n; c += a.chunk_rows) a.chunks[chunk++] = RouteChunk{e, row + c, min(a.chunk_rows, n - c), 0};
        counter[e] = row;
        row = end;
    }
    for (int c = all_chunks + tid; c < a.most_chunks; c += kGroupThreads) a.chunks[c] = RouteChunk{0, 0, 0, 0};
    if (tid == 0) *a.nchunks = all_chunks, *a.live_rows = all_rows;
    __syncthreads();

    auto place = [&](int r, int e, int x, int at) {
        const bool bad = (e & kBad) != 0;
        list_x[at] = bad ? -1 : x;
        list_of[at] = bad ? r | INT32_MIN : r;
    };
    int at[HOLD];
#pragma unroll
    for (int i = 0; i < HOLD; i++)
        if (held[i] >= 0) at[i] = atomicAdd(&counter[held[i] & (kBad - 1)], 1);
#pragma unroll
    for (int i = 0; i < HOLD; i++)
        if (held[i] >= 0) place(tid + i * kGroupThreads, held[i], from[i], at[i]);
    for (int r = tid + HOLD * kGroupThreads; r < a.routes; r += kGroupThreads) {
        const int e = expert_of(r);
        place(r, e, a.lhs ? a.lhs[r] : 0, atomicAdd(&counter[e & (kBad - 1)], 1));
    }
    __syncthreads();
    // Runs start at multiples of pad, and a counter is now where its run ends: -1 from there to the next multiple.
    if (a.pad > 1)
        for (int e = wave; e < E; e += kGroupThreads / kWave) {
            const int begin = counter[e], end = padded(begin);
            for (int i = begin + lane; i < end; i += kWave) list_x[i] = -1, list_of[i] = -1;
        }
    if constexpr (STAGED) {
        __syncthreads();
        // (lists in LDS and in memory have room for whole 16-byte pieces)
        for (int i = tid; i < (all_rows + 3) / 4; i += kGroupThreads) {
            reinterpret_cast<int4*>(a.route_x)[i] = reinterpret_cast<const int4*>(list_x)[i];
            reinterpret_cast<int4*>(a.route_of)[i] = reinterpret_cast<const int4*>(list_of)[i];
        }
    }
}

// LDS of a workgroup that groups.
inline size_t group_counter_bytes(const RouteGroupArgs& a) { return (size_t)(a.num_experts + 3) / 4 * 16; }
inline size_t group_staged_bytes(const RouteGroupArgs& a) { return group_counter_bytes(a) + (size_t)(a.most_rows + 3) / 4 * 32; }

}  // namespace aq
