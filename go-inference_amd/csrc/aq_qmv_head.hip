// lm_head: the vocabulary projection whose consumer wants a token, not 262 144 logits.
//
//   greedy   the projection with the argmax as its epilogue: each wavefront keeps the best packed (score, row)
//            of its rows and a small second kernel folds those; no logit is ever stored.  Replaces
//            rocm_mlx_q4_projection_greedy (go/engine/hip/kernels/quant/affine_projection_fused.hipinc:190-248).
//   scores   every row's (score, row) packed into 64 bits, the input of top-k sampling:
//            rocm_mlx_q4_projection_scores (:411-446).
//   top-k    the k largest packed values, sorted descending: what rocm_packed_topk
//            (go/engine/hip/kernels/sampling/topk.hipinc:45-84) yields per chunk, here per wavefront segment
//            and repeated until one segment is left.
//
// The streaming part is the dot2 body; only the epilogue differs.  best_score_kernel and pack_scores_kernel apply the same
// two epilogues to fp32 scores already in memory (shapes the dot2 kernels do not take, several rows).
#include "aq_qmv_body.h"

namespace aq {

template <int BITS, int R, int FUSE>
__global__ __launch_bounds__(4 * kWave) void qmv_head_kernel(const QmvArgs a) {
    qmv_dot2_body<BITS, 1, R, 4, 2, false, FUSE>(a, blockIdx.x);
}

typedef void (*QmvHeadKernel)(const QmvArgs);
struct QmvHeadEntry {
    int bits, fuse, rows;
    QmvHeadKernel fn;
};
#define AQ_HEAD(BITS, FUSE, R) {BITS, FUSE, R, qmv_head_kernel<BITS, R, FUSE>}
#define AQ_HEAD_SET(BITS) \
    AQ_HEAD(BITS, 3, 1), AQ_HEAD(BITS, 3, 2), AQ_HEAD(BITS, 3, 4), AQ_HEAD(BITS, 4, 1), AQ_HEAD(BITS, 4, 2), AQ_HEAD(BITS, 4, 4)
static const QmvHeadEntry kHeadTable[] = {AQ_HEAD_SET(4), AQ_HEAD_SET(8)};

static const QmvHeadEntry* find_head(int bits, int fuse, int rows) {
    for (const QmvHeadEntry& e : kHeadTable)
        if (e.bits == bits && e.fuse == fuse && e.rows == rows) return &e;
    return nullptr;
}

bool qmv_head_supported(int bits, int fuse, int rows) { return find_head(bits, fuse, rows) != nullptr; }

size_t qmv_head_partials(int N, int rows) { return (size_t)((N + rows * 4 - 1) / (rows * 4)) * 4; }

// Folds the per-wavefront maxima into best[0]: kHeadFoldGroups workgroups each fold a slice into their own
// slot, take a ticket, and the one that draws the last ticket folds the slots and zeroes the ticket counter
// again.  Sixty-four tickets on one address are cheap; one ticket per wavefront of the projection is not.
__global__ __launch_bounds__(256) void fold_best_kernel(const unsigned long long* __restrict__ partial, int count,
                                                        unsigned long long* fold, unsigned long long* __restrict__ best) {
    unsigned int* tickets = reinterpret_cast<unsigned int*>(fold);
    unsigned long long* slots = fold + 16;
    const int per_group = (count + kHeadFoldGroups - 1) / kHeadFoldGroups;
    const int begin = blockIdx.x * per_group;
    const int end = min(begin + per_group, count);
    unsigned long long mine = 0;
    constexpr int U = 4;
    for (int base = begin; base < end; base += 256 * U) {
        unsigned long long t[U];
#pragma unroll
        for (int u = 0; u < U; u++) {
            const int i = base + u * 256 + (int)threadIdx.x;
            // clamped, not predicated: reading a value twice does not change a maximum, and the loads stay
            // unconditional so that all of them are issued before the first is waited for
            t[u] = partial[min(i, end - 1)];
        }
#pragma unroll
        for (int u = 0; u < U; u++) mine = t[u] > mine ? t[u] : mine;
    }
    if (begin >= end) mine = 0;
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
        const unsigned long long other = __shfl_xor(mine, o, kWave);
        mine = other > mine ? other : mine;
    }
    __shared__ unsigned long long wave_best[4];
    __shared__ int last;
    if ((threadIdx.x & (kWave - 1)) == 0) wave_best[threadIdx.x >> 6] = mine;
    __syncthreads();
    if (threadIdx.x == 0) {
        unsigned long long b = wave_best[0];
        for (int i = 1; i < 4; i++) b = wave_best[i] > b ? wave_best[i] : b;
        __atomic_store_n(&slots[blockIdx.x], b, __ATOMIC_RELAXED);
        __threadfence();
        last = atomicAdd(tickets, 1u) == (unsigned int)kHeadFoldGroups - 1u;
    }
    __syncthreads();
    if (!last || threadIdx.x >= kWave) return;
    __threadfence();
    unsigned long long m = __atomic_load_n(&slots[threadIdx.x], __ATOMIC_RELAXED);  // kHeadFoldGroups == 64 lanes
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
        const unsigned long long other = __shfl_xor(m, o, kWave);
        m = other > m ? other : m;
    }
    if (threadIdx.x == 0) {
        best[0] = m;
        atomicExch(tickets, 0u);
    }
}

hipError_t qmv_head_launch(int bits, int fuse, int rows, const QmvArgs& a, hipStream_t stream) {
    const QmvHeadEntry* e = find_head(bits, fuse, rows);
    if (!e || a.M != 1) return hipErrorInvalidValue;
    const int rows_per_wg = rows * 4;
    const size_t lds = (size_t)a.K * 2;
    if (hipError_t rc = ensure_dynamic_lds(reinterpret_cast<const void*>(e->fn), (size_t)lds)) return rc;
    if (fuse == 3 && (!a.partial || !a.fold)) return hipErrorInvalidValue;
    hipLaunchKernelGGL(e->fn, dim3((unsigned)((a.N + rows_per_wg - 1) / rows_per_wg)), dim3(4 * kWave), lds, stream, a);
    hipError_t rc = hipGetLastError();
    if (rc != hipSuccess || fuse != 3) return rc;
    static_assert(kHeadFoldGroups == kWave, "the last workgroup reads one slot per lane");
    hipLaunchKernelGGL(fold_best_kernel, dim3(kHeadFoldGroups), dim3(256), 0, stream, a.partial,
                       (int)qmv_head_partials(a.N, rows), a.fold, reinterpret_cast<unsigned long long*>(a.y));
    return hipGetLastError();
}

// Greedy over a list of candidate rows (rocm_mlx_q4_projection_selected_greedy,
// go/engine/hip/kernels/quant/affine_projection_fused.hipinc:485-546).  The scores come from the gathered matvec: every
// candidate r is scored as one row of the window of `width` rows that starts at min(r, N - width) (an "expert" of a
// slab whose experts are one row apart), so a candidate costs width rows of weights and no kernel of its own is needed.
// windows: start[z] = first row of candidate z's window, -1 for an id outside [0, N).
__global__ __launch_bounds__(256) void selected_windows_kernel(const int32_t* __restrict__ rows, int count, int N, int width,
                                                               int32_t* __restrict__ start) {
    const int z = blockIdx.x * 256 + threadIdx.x;
    if (z >= count) return;
    const int r = rows[z];
    start[z] = (r >= 0 && r < N) ? min(r, N - width) : -1;
}
// pick: best[0] = max over the valid candidates with a finite score of pack(score, row); 0 when there is none.
__global__ __launch_bounds__(256) void selected_pick_kernel(const float* __restrict__ scores, const int32_t* __restrict__ rows,
                                                            const int32_t* __restrict__ start, int count, int width,
                                                            unsigned long long* __restrict__ best) {
    unsigned long long mine = 0;
    for (int z = threadIdx.x; z < count; z += 256) {
        const int e = start[z];
        if (e < 0) continue;
        const int r = rows[z];
        const float v = scores[(int64_t)z * width + (r - e)];
        if (isfinite(v)) {
            const unsigned long long p = pack_score_index(v, (uint32_t)r);
            mine = p > mine ? p : mine;
        }
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
        const unsigned long long other = __shfl_xor(mine, o, kWave);
        mine = other > mine ? other : mine;
    }
    __shared__ unsigned long long wave_best[4];
    if ((threadIdx.x & (kWave - 1)) == 0) wave_best[threadIdx.x >> 6] = mine;
    __syncthreads();
    if (threadIdx.x == 0) {
        unsigned long long b = wave_best[0];
        for (int i = 1; i < 4; i++) b = wave_best[i] > b ? wave_best[i] : b;
        best[0] = b;
    }
}
hipError_t selected_windows_launch(const int32_t* rows, int count, int N, int width, int32_t* start, hipStream_t stream) {
    hipLaunchKernelGGL(selected_windows_kernel, dim3((unsigned)((count + 255) / 256)), dim3(256), 0, stream, rows, count, N, width, start);
    return hipGetLastError();
}
hipError_t selected_pick_launch(const float* scores, const int32_t* rows, const int32_t* start, int count, int width,
                                unsigned long long* best, hipStream_t stream) {
    hipLaunchKernelGGL(selected_pick_kernel, dim3(1), dim3(256), 0, stream, scores, rows, start, count, width, best);
    return hipGetLastError();
}

hipError_t head_fold_launch(const unsigned long long* partial, int count, unsigned long long* fold, unsigned long long* best,
                            hipStream_t stream) {
    hipLaunchKernelGGL(fold_best_kernel, dim3(kHeadFoldGroups), dim3(256), 0, stream, partial, count, fold, best);
    return hipGetLastError();
}

// The epilogues over fp32 scores in memory.  scores: every value packed, a thread a value.
__global__ __launch_bounds__(256) void pack_scores_kernel(const float* __restrict__ scores, int N, const int32_t* suppress,
                                                          int suppress_count, unsigned long long* packed_out) {
    const int64_t row = (int64_t)blockIdx.y * N;
    for (int n = blockIdx.x * 256 + threadIdx.x; n < N; n += gridDim.x * 256) {
        const float v = scores[row + n];
        unsigned long long p = 0;
        if (isfinite(v) && !token_suppressed((uint32_t)n, suppress, suppress_count)) p = pack_score_index(v, (uint32_t)n);
        packed_out[row + n] = p;
    }
}

// argmax: grid.y = activation row.  One workgroup a row (ONE) stores the row's best itself; several meet in an atomic maximum
// on best[row], which starts at zero.  Atomics on one address are served one by one (about 12 ns each here): a workgroup
// for every 256 scores spent 36 us on 6 x 128201 scores and 60 us on 8 x 164024 in them, for 4 MB that are read in 3.  So at
// most kBestGroups of them per row, each thread with eight loads in flight; rows of up to kBestOneGroup scores in one
// workgroup of 1024 threads, which needs no launch that clears best (a longer row is more than one CU reads in the time of
// that launch: 128201 scores took it 18 us).  Whole greedy calls: 6 rows (128201 x 1152) 60.8 -> 29.6 us, 8 (164024 x 2048)
// 108.8 -> 54.7, 15 (91522 x 2048, 8 bit) 105.8 -> 65.3, 3 (36934 x 1536) 30.6 -> 27.0.
constexpr int kBestGroups = 32, kBestOneGroup = 16384;
// Suppressed tokens are bits of the workgroup's own scores, put down while the first scores are on their way.  (With the list looked
// through for every score that was a thread's largest so far, 2 x 16384 scores took 15.4 us with 3 entries, 70 with 40 and 453 with
// 300, beside 11 without a list; as bits 12.1, 12.3 and 12.5.)  Only rows of more than kBestBitsScores go through the list.
constexpr int kBestBitsScores = kBestOneGroup * kBestGroups;
enum { kNoList, kListAsBits, kListInMemory };
template <bool ONE, int LIST>
__global__ __launch_bounds__(ONE ? 1024 : 256) void best_score_kernel(const float* __restrict__ scores, int N, const int32_t* suppress,
                                                                     int suppress_count, unsigned long long* best) {
    constexpr int NT = ONE ? 1024 : 256, AHEAD = 8;
    const int m = blockIdx.y;
    const float* const row = scores + (int64_t)m * N;
    unsigned long long mine = 0;
    const int stride = (int)gridDim.x * NT;
    float v[AHEAD];
    auto fetch = [&](int64_t n0) {
#pragma unroll
        for (int i = 0; i < AHEAD; i++) v[i] = row[min(n0 + (int64_t)i * stride, (int64_t)N - 1)];
    };
    const int64_t first = (int64_t)blockIdx.x * NT + threadIdx.x;
    fetch(first);
    // bit: round * NT + thread, kBestOneGroup of them at the most
    __shared__ uint32_t gone[LIST == kListAsBits ? kBestOneGroup / 32 : 1];
    if constexpr (LIST == kListAsBits) {
        for (int i = threadIdx.x; i < kBestOneGroup / 32; i += NT) gone[i] = 0;
        __syncthreads();
        for (int i = threadIdx.x; i < suppress_count; i += NT) {
            const int s = suppress[i];
            if (s < 0 || s >= N) continue;
            const int round = s / stride, thread = s - round * stride - (int)blockIdx.x * NT;
            if (thread < 0 || thread >= NT) continue;
            const int bit = round * NT + thread;
            atomicOr(&gone[bit >> 5], 1u << (bit & 31));
        }
        __syncthreads();
    }
    int bit = threadIdx.x;
    for (int64_t n0 = first; n0 < N; n0 += (int64_t)stride * AHEAD, bit += NT * AHEAD) {
        uint32_t word[AHEAD] = {};
        if constexpr (LIST == kListAsBits)
#pragma unroll
            for (int i = 0; i < AHEAD; i++) word[i] = gone[min(bit + i * NT, kBestOneGroup - 1) >> 5];
#pragma unroll
        for (int i = 0; i < AHEAD; i++) {
            const int64_t n = n0 + (int64_t)i * stride;
            if (n >= N || !isfinite(v[i]) || (word[i] >> (bit & 31) & 1u)) continue;
            const unsigned long long p = pack_score_index(v[i], (uint32_t)n);
            if (p > mine && (LIST != kListInMemory || !token_suppressed((uint32_t)n, suppress, suppress_count))) mine = p;
        }
        if (n0 + (int64_t)stride * AHEAD < N) fetch(n0 + (int64_t)stride * AHEAD);
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
        const unsigned long long other = __shfl_xor(mine, o, kWave);
        mine = other > mine ? other : mine;
    }
    __shared__ unsigned long long wave_best[NT / kWave];
    if ((threadIdx.x & (kWave - 1)) == 0) wave_best[threadIdx.x >> 6] = mine;
    __syncthreads();
    if (threadIdx.x == 0) {
        unsigned long long b = wave_best[0];
        for (int i = 1; i < NT / kWave; i++) b = wave_best[i] > b ? wave_best[i] : b;
        if constexpr (ONE)
            best[m] = b;
        else if (b != 0)
            atomicMax(best + m, b);
    }
}

hipError_t pack_scores_launch(const float* scores, int M, int N, const int32_t* suppress, int suppress_count,
                              unsigned long long* packed, hipStream_t stream) {
    if (M <= 0 || N <= 0) return hipSuccess;
    int bx = (N + 255) / 256;
    if (bx > 1024) bx = 1024;
    hipLaunchKernelGGL(pack_scores_kernel, dim3((unsigned)bx, (unsigned)M), dim3(256), 0, stream, scores, N, suppress,
                       suppress_count, packed);
    return hipGetLastError();
}
bool best_score_clears(int N) { return N > 0 && N <= kBestOneGroup; }
hipError_t best_score_launch(const float* scores, int M, int N, const int32_t* suppress, int suppress_count, unsigned long long* best,
                             hipStream_t stream) {
    if (M <= 0 || N <= 0) return hipSuccess;
    typedef void (*BestKernel)(const float*, int, const int32_t*, int, unsigned long long*);
    static const BestKernel kBest[2][3] = {{best_score_kernel<false, kNoList>, best_score_kernel<false, kListAsBits>, best_score_kernel<false, kListInMemory>},
                                           {best_score_kernel<true, kNoList>, best_score_kernel<true, kListAsBits>, nullptr}};
    const bool one = best_score_clears(N);
    const int list = suppress_count == 0 ? kNoList : N <= kBestBitsScores ? kListAsBits : kListInMemory;
    hipLaunchKernelGGL(kBest[one][list], dim3(one ? 1u : (unsigned)min(kBestGroups, (N + 2047) / 2048), (unsigned)M), dim3(one ? 1024 : 256), 0, stream,
                       scores, N, suppress, suppress_count, best);
    return hipGetLastError();
}

// Maximum over the 64 lanes, unsigned: DPP folds inside each row of 16 lanes (a lane out of range reads 0,
// the identity), then the four row results meet through SGPRs.
__device__ __forceinline__ uint32_t wave_max_u32(uint32_t v) {
    v = max(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0xB1, 0xF, 0xF, true));
    v = max(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x4E, 0xF, 0xF, true));
    v = max(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x141, 0xF, 0xF, true));
    v = max(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x140, 0xF, 0xF, true));
    const uint32_t a = (uint32_t)__builtin_amdgcn_readlane((int)v, 0), b = (uint32_t)__builtin_amdgcn_readlane((int)v, 16);
    const uint32_t c = (uint32_t)__builtin_amdgcn_readlane((int)v, 32), d = (uint32_t)__builtin_amdgcn_readlane((int)v, 48);
    return max(max(a, b), max(c, d));
}

// One wavefront reduces kTopKSegment packed values to their top_k largest, sorted descending.  Every lane
// sorts its kTopKPerLane values in registers; then, top_k times, the wavefront takes the largest of the 64
// list heads (high words first, then the low words of the lanes that hold that high word) and the winning
// lane drops its head.  Entries past `count` read as 0, which is also the "no candidate" value.
__device__ __forceinline__ void topk_reduce_segment(const unsigned long long* in, int64_t count, int top_k, unsigned long long* out,
                                                    int64_t segment, int lane) {
    constexpr int V = kTopKPerLane;
    const int64_t begin = segment * kTopKSegment;
    if (begin >= count) return;  // whole wavefronts
    unsigned long long v[V];
#pragma unroll
    for (int j = 0; j < V; j++) {
        const int64_t i = begin + j * kWave + lane;
        v[j] = i < count ? in[i] : 0ull;
    }
    // bitonic network over the lane's own values, fully unrolled: descending order
#pragma unroll
    for (int width = 2; width <= V; width <<= 1) {
#pragma unroll
        for (int stride = width >> 1; stride > 0; stride >>= 1) {
#pragma unroll
            for (int i = 0; i < V; i++) {
                const int j = i ^ stride;
                if (j > i) {
                    const bool descending = (i & width) == 0;
                    const unsigned long long a = v[i], b = v[j];
                    const bool swap = descending ? a < b : a > b;
                    v[i] = swap ? b : a;
                    v[j] = swap ? a : b;
                }
            }
        }
    }
    unsigned long long mine = 0;
    for (int it = 0; it < top_k; it++) {
        const uint32_t hi = (uint32_t)(v[0] >> 32), lo = (uint32_t)v[0];
        const uint32_t best_hi = wave_max_u32(hi);
        const uint32_t best_lo = wave_max_u32(hi == best_hi ? lo : 0u);
        const unsigned long long best = ((unsigned long long)best_hi << 32) | best_lo;
        if (best == 0) break;  // nothing but "no candidate" left; uniform over the wavefront
        const unsigned long long holders = __ballot(v[0] == best);
        if (lane == __ffsll((long long)holders) - 1) {  // equal values: one lane at a time gives its copy
#pragma unroll
            for (int j = 0; j + 1 < V; j++) v[j] = v[j + 1];
            v[V - 1] = 0;
        }
        if (lane == it) mine = best;
    }
    if (lane < top_k) out[segment * top_k + lane] = mine;
}

// A round of the segment-by-segment reduction.
__global__ __launch_bounds__(256) void packed_topk_kernel(const unsigned long long* __restrict__ in, int64_t count, int top_k,
                                                          unsigned long long* __restrict__ out) {
    topk_reduce_segment(in, count, top_k, out, (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6), threadIdx.x & (kWave - 1));
}

// Threshold path, for inputs of many segments: two launches.  The top_k-th largest of any set of maxima over disjoint parts of
// the input is a value T that at least top_k entries reach (the maxima themselves), so the top_k largest entries all lie among
// the entries >= T.
//   lists   a workgroup takes 256 * V entries, finds T from the maxima of its 256 threads and lists the entries >= T, a little
//           over top_k of them for scores that are not arranged by rank, beside the maxima of its four wavefronts;
//   merge   T over all of those maxima leaves a little over top_k entries of the lists, which one workgroup orders by counting.
// When a list overflows or more than kTopKCandidates entries are left (long runs of equal scores, an input sorted by score) the
// second launch runs the segment-by-segment reduction instead, all its rounds: as launches of their own, which left at once where
// there was nothing to do, the later ones took 1.6 us each of every call.
// Bound: latency of the two launches (2 MB are read in a fraction of one).  Maxima, filter and finish as three launches -> here (us,
// the best 40 / 64): 50220 entries 15.4 / 13.5 -> 11.0 / 11.0, 262144 13.6 / 16.3 -> 10.1 / 12.0, sorted by score 53.5 / 70.6 ->
// 22.8 / 69.4.
// V is the largest of 16, 4, 1 that leaves at least top_k wavefronts with a maximum each.
// Head of the threshold path's scratch in 8-byte entries: the tickets of the tree's nodes, 4 bytes each (at most 1024 segments in
// nodes of 16 lists or more: 64 + 4 + 1).
constexpr int kTopKHeader = 40;
constexpr int kTopKListMax = 2 * kTopKMax;             // entries a list holds
static_assert(kTopKMax <= kTopKSegment / 16 && kTopKThresholdSegments <= 1024 && 64 + 4 + 1 <= 2 * kTopKHeader && 2 * kTopKHeader <= 256, "tickets");
static_assert(kTopKMax <= kWave, "at least top_k lanes hold a maximum");

// A t that at least top_k of the keys (SV a lane, zero where there is none) reach, and few more unless it is the largest such: built
// bit by bit from the top, every count one ballot.  The smallest of the lanes' maxima is reached by 64 of them, so the bits that
// it shares with the largest are t's.  The last bits are only asked for where the scores agree in the others.
constexpr int kTopKThresholdShift = 12;

template <int SV>
__device__ __forceinline__ uint32_t topk_threshold_key(const uint32_t (&key)[SV], int top_k) {
    uint32_t m = key[0];
#pragma unroll
    for (int j = 1; j < SV; j++) m = max(m, key[j]);
    const uint32_t most = wave_max_u32(m), least = ~wave_max_u32(~m);
    const int shared = most == least ? 32 : __builtin_clz(most ^ least);  // leading bits
    uint32_t t = shared == 0 ? 0u : most & (0xffffffffu << (32 - shared));
    int reached = SV * kWave;  // (or more than anyone asks for, where t is what all of them share)
    auto try_bit = [&](int bit) {
        const uint32_t trial = t | (1u << bit);
        int reach = 0;
#pragma unroll
        for (int j = 0; j < SV; j++) reach += __popcll(__ballot(key[j] >= trial));
        if (reach >= top_k) t = trial, reached = reach;
    };
    int bit = 31 - shared;
    for (; bit >= kTopKThresholdShift; bit--) try_bit(bit);
    if (__builtin_expect(t != 0 && reached > max(top_k + 8, 48), 0))
        for (; bit >= 0; bit--) try_bit(bit);
    return t;
}

// lists: [lists][kTopKListMax]; sizes: entries of each (more than kTopKListMax: it has overflowed); keys: the high words of the
// wavefronts' maxima
template <int V>
__global__ __launch_bounds__(256) void topk_lists_kernel(const unsigned long long* __restrict__ in, int64_t count, int top_k,
                                                         unsigned long long* __restrict__ lists, uint32_t* __restrict__ sizes,
                                                         uint32_t* __restrict__ keys, uint32_t* tickets) {
    __shared__ uint32_t thread_key[256];
    __shared__ uint32_t filled;
    const int tid = threadIdx.x, lane = tid & (kWave - 1);
    const int64_t begin = (int64_t)blockIdx.x * (256 * V);
    if (blockIdx.x == 0 && tid < kTopKHeader * 2) tickets[tid] = 0;
    if (tid == 0) filled = 0;
    unsigned long long v[V], m = 0;
#pragma unroll
    for (int j = 0; j < V; j++) {
        const int64_t i = begin + j * 256 + tid;
        v[j] = i < count ? in[i] : 0ull;
    }
#pragma unroll
    for (int j = 0; j < V; j++) m = v[j] > m ? v[j] : m;
    thread_key[tid] = (uint32_t)(m >> 32);
    const uint32_t wave_key = wave_max_u32((uint32_t)(m >> 32));
    if (lane == 0) keys[blockIdx.x * 4 + (tid >> 6)] = wave_key;
    __syncthreads();
    uint32_t key[4];
#pragma unroll
    for (int j = 0; j < 4; j++) key[j] = thread_key[j * kWave + lane];
    const unsigned long long t = (unsigned long long)topk_threshold_key<4>(key, top_k) << 32;
    unsigned long long mask[V];
    int total = 0;
#pragma unroll
    for (int j = 0; j < V; j++) {
        mask[j] = __ballot(v[j] >= t && v[j] != 0);
        total += __popcll(mask[j]);
    }
    uint32_t base = 0;
    if (lane == 0 && total) base = atomicAdd(&filled, (uint32_t)total);
    base = (uint32_t)__builtin_amdgcn_readfirstlane((int)base);
    const unsigned long long below = (1ull << lane) - 1;
#pragma unroll
    for (int j = 0; j < V; j++) {
        const uint32_t pos = base + (uint32_t)__popcll(mask[j] & below);
        if (((mask[j] >> lane) & 1) && pos < (uint32_t)kTopKListMax) lists[(int64_t)blockIdx.x * kTopKListMax + pos] = v[j];
        base += (uint32_t)__popcll(mask[j]);
    }
    __syncthreads();
    if (tid == 0) sizes[blockIdx.x] = filled;
}

// Workgroup 0 merges; the others are there for the inputs that go through the tree, which all find out in the same way.
// The candidates are distinct unless the input repeats a value, so an entry's place in the output is the number of candidates
// above it (equal values take consecutive places).
constexpr int kMergeThreads = 1024, kTreeWaves = 4;  // (the tree runs on a few wavefronts of many workgroups)
template <int SV>
__global__ __launch_bounds__(kMergeThreads) void topk_merge_kernel(const unsigned long long* __restrict__ in, int64_t count, int top_k,
                                                                   const unsigned long long* __restrict__ lists,
                                                                   const uint32_t* __restrict__ sizes, const uint32_t* __restrict__ keys,
                                                                   int nlists, unsigned long long* __restrict__ out,
                                                                   unsigned long long* tree, uint32_t* tickets) {
    constexpr int WAVES = kMergeThreads / kWave;
    constexpr int PER_WAVE = SV * 16 / WAVES;  // lists a wavefront takes (16 SV of them at the most)
    __shared__ unsigned long long c[kTopKCandidates];
    __shared__ uint32_t filled;
    const int tid = threadIdx.x, lane = tid & (kWave - 1), wave = tid >> 6;
    if (tid == 0) filled = 0;
    uint32_t key[SV], size[PER_WAVE];
#pragma unroll
    for (int j = 0; j < SV; j++) key[j] = j * kWave + lane < 4 * nlists ? keys[j * kWave + lane] : 0u;
    unsigned long long v[PER_WAVE];  // the first 64 entries (past a list's size: unset); few lists have more
#pragma unroll
    for (int i = 0; i < PER_WAVE; i++) {
        const int l = wave + i * WAVES;
        size[i] = l < nlists ? sizes[l] : 0u;
        v[i] = l < nlists ? lists[(int64_t)l * kTopKListMax + lane] : 0ull;
    }
    __syncthreads();
    const unsigned long long t = (unsigned long long)topk_threshold_key<SV>(key, top_k) << 32;
#pragma unroll
    for (int i = 0; i < PER_WAVE; i++) {
        if (size[i] > (uint32_t)kTopKListMax) {  // an overflow, seen by every workgroup alike
            if (lane == 0) atomicAdd(&filled, (uint32_t)kTopKCandidates + 1);
            continue;
        }
        for (uint32_t from = 0; from < size[i]; from += kWave) {
            if (from) v[i] = lists[(int64_t)(wave + i * WAVES) * kTopKListMax + from + lane];
            const unsigned long long mask = __ballot(from + lane < size[i] && v[i] >= t);
            if (mask == 0) continue;
            uint32_t base = 0;
            if (lane == 0) base = atomicAdd(&filled, (uint32_t)__popcll(mask));
            base = (uint32_t)__builtin_amdgcn_readfirstlane((int)base);
            const uint32_t pos = base + (uint32_t)__popcll(mask & ((1ull << lane) - 1));
            if (((mask >> lane) & 1) && pos < (uint32_t)kTopKCandidates) c[pos] = v[i];
        }
    }
    __syncthreads();
    const uint32_t n = filled;
    if (n > (uint32_t)kTopKCandidates) {
        // A tree of lists: every wavefront reduces its segment, and the one that completes the children of a node (as many
        // lists as fill a segment) reduces those too and goes on from there.  Every list has a place of its own.
        const int fan = kTopKSegment / top_k;
        int64_t left = (count + kTopKSegment - 1) / kTopKSegment, at = (int64_t)blockIdx.x * kTreeWaves + wave;
        if (wave >= kTreeWaves || at >= left) return;
        topk_reduce_segment(in, count, top_k, tree, at, lane);
        while (true) {
            const int64_t node = at / fan, first = node * fan, nodes = (left + fan - 1) / fan;
            const int children = (int)(left - first < fan ? left - first : fan);
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "agent");  // this wavefront's list is visible before its ticket is
            uint32_t before = 0;
            if (lane == 0) before = atomicAdd(tickets + node, 1u);
            if (__builtin_amdgcn_readfirstlane((int)before) + 1 != children) return;
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
            unsigned long long* const dst = nodes == 1 ? out : tree + left * top_k;
            topk_reduce_segment(tree + first * top_k, (int64_t)children * top_k, top_k, dst + node * top_k, 0, lane);
            if (nodes == 1) return;
            tree = dst;
            tickets += nodes;
            left = nodes;
            at = node;
        }
    }
    if (blockIdx.x != 0) return;
    for (uint32_t idx = tid; idx < n; idx += kMergeThreads) {
        const unsigned long long mine = c[idx];
        int rank = 0;
#pragma unroll 8
        for (uint32_t o = 0; o < n; o++) {
            const unsigned long long other = c[o];
            rank += (other > mine || (other == mine && o < idx)) ? 1 : 0;
        }
        if (rank < top_k) out[rank] = mine;
    }
    if ((uint32_t)tid >= n && tid < top_k) out[tid] = 0ull;  // fewer candidates than top_k
}

static int64_t topk_segments(int64_t count) { return (count + kTopKSegment - 1) / kTopKSegment; }

// Entries a lane takes on the threshold path, 0 when the input goes segment by segment: the path needs at least
// top_k maxima and a wavefront keeps the whole list of maxima in registers.
static int topk_threshold_per_lane(int64_t count, int top_k) {
    if (count <= kTopKSegment) return 0;
    for (int v : {16, 4, 1}) {
        const int64_t pieces = (count + kWave * v - 1) / (kWave * v);
        if (pieces >= top_k && pieces <= kTopKThresholdSegments) return v;
    }
    return 0;
}

static int64_t topk_lists(int64_t count, int top_k) {
    const int64_t entries = 256 * topk_threshold_per_lane(count, top_k);
    return (count + entries - 1) / entries;
}

// Entries of the tree of lists (topk_merge_kernel; the last list is the call's output).
static int64_t topk_tree_entries(int64_t count, int top_k) {
    const int64_t fan = kTopKSegment / top_k;
    int64_t total = 0;
    for (int64_t lists = topk_segments(count); lists > 1; lists = (lists + fan - 1) / fan) total += lists * top_k;
    return total;
}

size_t packed_topk_scratch_entries(int64_t count, int top_k) {
    if (count <= kTopKSegment) return 0;
    // first round's output, then the second round's beside it (every later round is smaller)
    const int64_t c1 = topk_segments(count) * top_k;
    const int64_t c2 = c1 > kTopKSegment ? topk_segments(c1) * top_k : 0;
    if (topk_threshold_per_lane(count, top_k))
        return (size_t)(topk_tree_entries(count, top_k) + kTopKHeader + kTopKThresholdSegments + topk_lists(count, top_k) * kTopKListMax);
    return (size_t)(c1 + c2);
}

hipError_t packed_topk_launch(const unsigned long long* in, int64_t count, int top_k, unsigned long long* out,
                              unsigned long long* scratch, hipStream_t stream) {
    if (top_k <= 0 || top_k > kTopKMax || count <= 0) return hipErrorInvalidValue;
    const int64_t first = topk_segments(count);
    const int64_t c1 = first * top_k;
    unsigned long long* bufs[2] = {scratch, scratch + c1};
    int which = 0;
    const unsigned long long* src = in;
    int64_t n = count;
    if (const int per_lane = topk_threshold_per_lane(count, top_k)) {
        unsigned long long* const extra = scratch + topk_tree_entries(count, top_k);
        uint32_t* const tickets = reinterpret_cast<uint32_t*>(extra);
        uint32_t* const keys = reinterpret_cast<uint32_t*>(extra + kTopKHeader);
        uint32_t* const sizes = keys + kTopKThresholdSegments;
        unsigned long long* const lists = extra + kTopKHeader + kTopKThresholdSegments;
        const int nlists = (int)topk_lists(count, top_k);
        hipLaunchKernelGGL(per_lane == 16 ? topk_lists_kernel<16> : per_lane == 4 ? topk_lists_kernel<4> : topk_lists_kernel<1>,
                           dim3((unsigned)nlists), dim3(256), 0, stream, in, count, top_k, lists, sizes, keys, tickets);
        hipLaunchKernelGGL(nlists <= 64 ? topk_merge_kernel<4> : topk_merge_kernel<kTopKThresholdSegments / kWave>,
                           dim3((unsigned)((first + kTreeWaves - 1) / kTreeWaves)), dim3(kMergeThreads), 0, stream, in, count, top_k, lists, sizes,
                           keys, nlists, out, scratch, tickets);
        return hipGetLastError();
    }
    while (true) {
        const int64_t segments = topk_segments(n);
        unsigned long long* dst = segments == 1 ? out : bufs[which];
        hipLaunchKernelGGL(packed_topk_kernel, dim3((unsigned)((segments + 3) / 4)), dim3(256), 0, stream, src, n, top_k, dst);
        hipError_t rc = hipGetLastError();
        if (rc != hipSuccess || segments == 1) return rc;
        src = dst;
        n = segments * top_k;
        which ^= 1;
    }
}

// Temperature / top-p sampling over the packed top-k list (rocm_packed_topk_sample,
// go/engine/hip/kernels/sampling/topk.hipinc:86-191; score decode and softcap kernels/common/numeric.hipinc:95-110).
// The reference runs the whole thing on one thread and evaluates exp() of every candidate in each of its four
// passes; here each of up to 128 threads evaluates its candidate's weight once (tanh and exp in double are the
// cost), thread 0 adds them once in list order, as the reference does, so every sum rounds the same way, and the
// threads compare against that running sum side by side.  out[0] = 0 when nothing can be sampled.
constexpr int kSampleMax = 128;

__device__ __forceinline__ double sample_score(unsigned long long packed, double softcap) {
    const uint32_t key = (uint32_t)(packed >> 32);
    const double score = (double)__uint_as_float((key & 0x80000000u) ? key ^ 0x80000000u : ~key);
    return softcap > 0.0 ? tanh(score / softcap) * softcap : score;
}

__global__ __launch_bounds__(kSampleMax) void packed_topk_sample_kernel(const unsigned long long* __restrict__ in,
                                                                        int top_k, float raw_temperature, float raw_top_p,
                                                                        float softcap_f, double draw,
                                                                        unsigned long long* __restrict__ out) {
    __shared__ unsigned long long vals[kSampleMax];
    __shared__ double wts[kSampleMax];
    __shared__ double prefix[kSampleMax];
    __shared__ double total_s;
    __shared__ int bad, limit_s, kept_s, pick_s;
    const int t = threadIdx.x;
    vals[t] = t < top_k ? in[t] : 0ull;
    if (t == 0) {
        bad = 0;
        limit_s = top_k;
        kept_s = 0;
        pick_s = kSampleMax;
    }
    __syncthreads();
    int first_valid = top_k;  // the same scan on every thread: the branches below are uniform
    for (int i = 0; i < top_k; ++i)
        if (vals[i] != 0ull) {
            first_valid = i;
            break;
        }
    unsigned long long result = 0ull;
    bool sample = false;
    double temperature = 1.0, top_p = 1.0;
    if (first_valid < top_k) {
        if (raw_temperature <= 0.0f && raw_top_p <= 0.0f) {
            result = vals[first_valid];  // greedy
        } else {
            temperature = raw_temperature == 0.0f ? 1.0 : (double)raw_temperature;
            top_p = raw_top_p == 0.0f ? 1.0 : (double)raw_top_p;
            sample = temperature > 0.0 && top_p > 0.0 && top_p <= 1.0;
        }
    }
    if (!sample) {
        if (t == 0) out[0] = result;
        return;
    }
    const double softcap = (double)softcap_f;
    const bool valid = t >= first_valid && t < top_k && vals[t] != 0ull;
    const double score = valid ? sample_score(vals[t], softcap) / temperature : 0.0;
    prefix[t] = score;  // (the first valid one's is every thread's maximum: tanh once, not twice in turn)
    __syncthreads();
    wts[t] = valid ? exp(score - prefix[first_valid]) : 0.0;
    if (valid && !isfinite(wts[t])) bad = 1;  // any non-finite weight: nothing is sampled
    __syncthreads();
    // The reference's four passes all add the same weights in the same order from 0.0: its total, its nucleus
    // cumulative, its selected total and its draw cumulative are entries of ONE running sum.  Thread 0 forms that
    // sum once; the comparisons against it are independent and every thread does its own.
    if (t == 0) {
        double run = 0.0;  // holes carry weight 0.0, and x + 0.0 is x: no branch in the chain of adds
#pragma unroll 8
        for (int i = 0; i < top_k; ++i) {
            run += wts[i];
            prefix[i] = run;
        }
        total_s = run;
    }
    __syncthreads();
    const double total = total_s;
    if (bad || !(total > 0.0) || !isfinite(total)) {
        if (t == 0) out[0] = 0ull;
        return;
    }
    if (top_p < 1.0 && valid && prefix[t] / total >= top_p) atomicMin(&limit_s, t + 1);
    __syncthreads();
    const int limit = limit_s;
    if (valid && t < limit) atomicMax(&kept_s, t);  // the last candidate inside the nucleus
    __syncthreads();
    const int kept = kept_s;
    const double selected_total = prefix[kept];
    if (!(selected_total > 0.0) || !isfinite(selected_total)) {
        if (t == 0) out[0] = 0ull;
        return;
    }
    if (draw < 0.0) draw = 0.0;
    if (draw >= 1.0) draw = 0x1.fffffffffffffp-1;  // the double below 1
    const double target = draw * selected_total;
    if (valid && t < limit && target <= prefix[t]) atomicMin(&pick_s, t);
    __syncthreads();
    if (t == 0) out[0] = vals[pick_s < kSampleMax ? pick_s : kept];
}

hipError_t packed_topk_sample_launch(const unsigned long long* in, int top_k, float temperature, float top_p, float softcap,
                                     double draw, unsigned long long* out, hipStream_t stream) {
    if (top_k <= 0 || top_k > kSampleMax) return hipErrorInvalidValue;
    hipLaunchKernelGGL(packed_topk_sample_kernel, dim3(1), dim3(kSampleMax), 0, stream, in, top_k, temperature, top_p, softcap,
                       draw, out);
    return hipGetLastError();
}

}  // namespace aq
