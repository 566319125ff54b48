// Expert slabs of 4-bit codes in groups of 32, 64 and 128: routes grouped by expert (aq_moe_group.hip), a workgroup for up to 48 routes
// of one expert by 256 of its weight rows.
//
// The operands are those of aq_qmm_half.hip (scale * (code - 8) exact in fp16, rows of x and of the weights brought into fp16's range
// by powers of two, the affine term as a bf16 product of group sums); what differs is how a tile is cut and fed.
//
// A prompt of 512 tokens gives an expert of 128 thirty-two routes, as many more as fewer, so that 32-row tiles read and expand the
// weights of half of the experts twice, and 64-row tiles multiply mostly rows that are not there.  Here rows come in blocks of 16
// (v_mfma_f32_16x16x32): a workgroup runs the loop of as many as its chunk fills, 1, 2 or 3.  Three are what leaves three workgroups
// to a CU (168 registers; groups of 32 two), and 128 experts times 6 strips are then one round of them.  512 tokens, 2816 / 704: gate
// and up 115 -> 90 us, down 72 -> 62, the block 233 -> 185.
//
// A wavefront owns 64 weight rows over all of K.  Nobody shares its codes, so they go from memory into registers, a line of 256 codes of
// each row ahead of its use; lane (n, q) then holds codes 32 q .. 32 q + 31 of either half of row n, and K is multiplied in that order
// (x is written in it).  Scales and biases of 16 groups are one load each, four of a row to a lane: the affine product takes
// them as they lie, the scales are handed round by ds_bpermute.  x goes through LDS, two steps of 256 codes, from where the pass over it
// left each row: that runs over the rows of x as the caller has them, once each however many routes read it, and beside the
// list of routes (per route and behind the list: 7.8 + 13.9 us of gate and up -> 8.8).
//
// Bound (gate and up above): 391 MB past the L2s, 285 of them the weights (the lines of the scales are fetched again in every segment),
// in 88 us, 4.4 TB/s; vector issue 64 % of SIMD cycles, matrix cores 21 %, wavefronts wait 26 % of theirs.  The first 10 us of a round
// are its first lines on their way, of all tiles at once.  Codes with the non-temporal hint: 194 -> 198 us the block.
#include "aq_device.h"
#include "aq_fp16_operands.h"
#include "aq_kernels.h"
#include "aq_lds_copy.h"
#include "aq_moe_group.h"
#include "aq_qmm.h"

#include <type_traits>

namespace aq {

namespace {

typedef _Float16 f16x2_t __attribute__((ext_vector_type(2)));
typedef _Float16 f16x8_t __attribute__((ext_vector_type(8)));
typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2_t __attribute__((ext_vector_type(2)));
typedef uint32_t u32_at2_t __attribute__((aligned(2)));
typedef uint32_t u32x2_at2_t __attribute__((ext_vector_type(2), aligned(2)));

constexpr int kPiece = 128;           // codes of a row that four lanes hold 16 bytes of each
constexpr int kStep = 2 * kPiece;     // codes of a step of the loop: a 128-byte line of a row
constexpr int kElements = 16;         // elements of a row of scales that four lanes hold four of each: a segment
constexpr int kThreads = 256, kWaves = kThreads / kWave;
constexpr int kCols = kWaves * 64;
constexpr int kStage = 16 * kStep * 2;  // bytes of 16 rows of x

// A load at a uniform base and a 32-bit offset of the lane.  (The offset is hidden from the compiler, which would carry a 64-bit address
// per load through the loop: 36 registers of 154 with one row block.)
__device__ __forceinline__ uint32_t hidden(uint32_t v) {
    asm volatile("" : "+v"(v));
    return v;
}
typedef const __attribute__((address_space(1))) uint8_t* global_t;
template <typename T>
__device__ __forceinline__ T load_at(global_t base, uint32_t off) {
    return *reinterpret_cast<const __attribute__((address_space(1))) T*>(base + hidden(off));
}
// largest finite magnitude (bf16 bits) of the halves of a word and of `most`
__device__ __forceinline__ uint32_t most_of(uint32_t most, uint32_t w) {
    const uint32_t lo = w & 0x7fffu, hi = w >> 16 & 0x7fffu;
    return max(most, max(lo < 0x7f80u ? lo : 0u, hi < 0x7f80u ? hi : 0u));
}

}  // namespace

// ---- pass over x ----------------------------------------------------------------------------------------------------
// A wavefront a row.  xf: [rows][K up to a multiple of 256] fp16, x * 2^e with e per row, the eight values of a word of codes in the
// order in which they are expanded; xs: [rows][groups up to a multiple of 16] the group's sum times 2^e as two bf16 in a word;
// rs: [rows] 2^-e.  Padding is zeros.  from: the row of x that row i is (null: i).
// Workgroup 0 of a launch of 1024 threads puts the list of routes together meanwhile (a list too long for that has a launch of its
// own, `first` is 0 then): neither needs the other.  512 tokens through 128 experts: 5.8 us of list and 6 of x as two launches.
constexpr int kPrepThreads = kGroupThreads;
constexpr size_t kListLds = 40 * 1024;  // of a list in the same launch: three workgroups of x a CU beside it
template <int GRP>
__global__ __launch_bounds__(kPrepThreads) void qmmr_prep_kernel(const uint16_t* __restrict__ x, uint16_t* __restrict__ xf, uint32_t* __restrict__ xs,
                                                                 float* __restrict__ rs, int rows, int K, const int32_t* __restrict__ from, int x_rows,
                                                                 const RouteGroupArgs lists, int first) {
    constexpr int HOLD = 8;
    if ((int)blockIdx.x < first) {
        extern __shared__ __attribute__((aligned(16))) int32_t counter[];
        group_routes<true>(lists, counter);
        return;
    }
    const int row = ((int)blockIdx.x - first) * (kPrepThreads / kWave) + (int)threadIdx.x / kWave, lane = threadIdx.x & (kWave - 1);
    if (row >= rows) return;
    const int pieces = K / 8, padded = (K + kStep - 1) / kStep * (kStep / 8), all = (K + kElements * GRP - 1) / (kElements * GRP) * (kElements * GRP / 8);
    const int src = from ? from[row] : row;
    const uint16_t* const xrow = x + (int64_t)(src < 0 || src >= x_rows ? 0 : src) * K;  // (out of range: the row is not read)
    uint4 hold[HOLD];
    auto fetch = [&](int p0) {
#pragma unroll
        for (int i = 0; i < HOLD; i++) {
            hold[i] = make_uint4(0u, 0u, 0u, 0u);
            const int p = p0 + i * kWave + lane;
            if (p < pieces) hold[i] = *reinterpret_cast<const uint4*>(xrow + p * 8);
        }
    };
    uint32_t mag = 0;
    for (int p0 = 0; p0 < pieces; p0 += HOLD * kWave) {
        fetch(p0);
#pragma unroll
        for (int i = 0; i < HOLD; i++) mag = most_of(most_of(most_of(most_of(mag, hold[i].x), hold[i].y), hold[i].z), hold[i].w);
    }
    mag = max_lanes<1>(mag);
    const int e = exponent_shift(mag, 14);
    const float up = pow2f(e);
    if (lane == 0) rs[row] = pow2f(-e);
    uint16_t* const to = xf + (int64_t)row * padded * 8;
    uint32_t* const sums = xs + (int64_t)row * (all * 8 / GRP);
    for (int p0 = 0; p0 < all; p0 += HOLD * kWave) {
        if (pieces > HOLD * kWave) fetch(p0);
#pragma unroll
        for (int i = 0; i < HOLD; i++) {
            const int p = p0 + i * kWave + lane;
            if (p0 + i * kWave >= all) break;
            const uint32_t w[4] = {hold[i].x, hold[i].y, hold[i].z, hold[i].w};
            float sx = 0.0f;
#pragma unroll
            for (int c = 0; c < 4; c++) sx = dot2_bf16(w[c], 0x3F803F80u, sx);
#pragma unroll
            for (int o = 1; o < GRP / 8; o <<= 1) sx += __shfl_xor(sx, o, kWave);
            if (p < all && p % (GRP / 8) == 0) {
                const float scaled = sx * up;
                const uint32_t hi = f32_to_bf16_bits(scaled), lo = f32_to_bf16_bits(scaled - bf16_bits_to_f32(hi));
                sums[p / (GRP / 8)] = hi | lo << 16;
            }
            if (p < padded) {
                _Float16 h[8];
#pragma unroll
                for (int c = 0; c < 4; c++) {
                    h[2 * c] = (_Float16)(bf16_bits_to_f32(w[c] & 0xffffu) * up);
                    h[2 * c + 1] = (_Float16)(bf16_bits_to_f32(w[c] >> 16) * up);
                }
                *reinterpret_cast<f16x8_t*>(to + p * 8) = f16x8_t{h[0], h[4], h[1], h[5], h[2], h[6], h[3], h[7]};
            }
        }
    }
}

// ---- main kernel ----------------------------------------------------------------------------------------------------
template <int GRP>
__global__ __launch_bounds__(kThreads, GRP == 32 ? 2 : 3) void qmmr_kernel(const QmmRouteArgs a) {
    __shared__ __align__(16) uint8_t stage[2 * (kRouteRows / 16) * kStage];
    __shared__ __align__(16) uint32_t sums[kRouteRows * kElements];  // of x, of a segment: [block of rows][quarter q][row][four of them]
    __shared__ int32_t route[kRouteRows];                    // per row of the tile: its route,
    __shared__ uint32_t x_at[kRouteRows], sum_at[kRouteRows];  // where its row of xf and of xs begins, in bytes,
    __shared__ float down[kRouteRows];                       // and the inverse power of two of that row
    constexpr int SPS = kElements * GRP / kStep;             // steps of a segment
    // Workgroups are dealt to the XCDs round-robin: the strips of a chunk, which read the same x, are on one, next to each other.
    const int in_run = (int)blockIdx.x >> 3, round = in_run / a.strips, chunk = round * 8 + ((int)blockIdx.x & 7);
    if (chunk >= a.most_chunks) return;
    const RouteChunk ch = a.chunks[chunk];
    const int count = __builtin_amdgcn_readfirstlane(ch.count);
    if (count == 0) return;  // behind the end of the list
    const int tid = threadIdx.x, lane = tid & (kWave - 1), wave = __builtin_amdgcn_readfirstlane(tid / kWave);
    const int n = lane & 15, q = lane >> 4;
    const int K = a.K, N = a.N, pair = a.pair;
    // what thread i < kRouteRows puts into the lists (a row out of range: any row of xf, its outputs are zeros)
    const int at_route = __builtin_amdgcn_readfirstlane(ch.first) + min(tid, count - 1);
    const int my_route = a.route_of[at_route];
    const int my_x = max(a.by_route ? my_route & INT32_MAX : a.route_x[at_route], 0);

    const int n0 = (in_run - round * a.strips) * (pair ? kCols / 2 : kCols);
    auto uniform = [](const void* p) {
        const uint64_t u = reinterpret_cast<uint64_t>(p);
        const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)u), hi = __builtin_amdgcn_readfirstlane((uint32_t)(u >> 32));
        return (global_t)((uint64_t)hi << 32 | lo);
    };
    global_t wt[2], st[2], bt[2];  // the tile's first weight row, gate and up (the same where there is one matrix)
#pragma unroll
    for (int i = 0; i < 2; i++) {
        const int64_t first = (int64_t)__builtin_amdgcn_readfirstlane(ch.expert) * a.expert_rows + n0 + (i && pair ? a.row_base2 : a.row_base);
        wt[i] = uniform(a.w + first * (K / 8));
        st[i] = uniform(a.s + first * (K / GRP));
        bt[i] = uniform(a.b + first * (K / GRP));
    }
    const int pieces = (K + kPiece - 1) / kPiece, steps = (K + kStep - 1) / kStep;
    const int groups = K / GRP, segments = (groups + kElements - 1) / kElements;
    const uint32_t row_bytes = (uint32_t)K / 2, sb_bytes = (uint32_t)groups * 2;

    // column block cg of the wavefront: its matrix, and its weight row i counted from the tile's first
    auto second = [&](int cg) { return pair && cg >= 2; };
    auto row = [&](int cg, int i) { return min((uint32_t)(wave * (pair ? 32 : 64) + i) + (uint32_t)((pair ? cg & 1 : cg) * 16), (uint32_t)(N - 1 - n0)); };
    // Codes of step c of column blocks 2 cp and 2 cp + 1: a line of each row.  A load takes whole lines of eight rows (16 bytes of
    // lane (n, q): row n % 8, pieces q and 4 + q for lanes below and from n = 8 on; the second load rows 8 on): the L1 charges
    // a load by the line, and half a line of sixteen rows at a time was 512 of the 1150 clocks that a wavefront's step cost it.
    // in_order() then hands over between the lanes n and n ^ 8: half h of row n is word h of lane (n, q).
    u32x4_t cw[2][2][2];  // [pair of column blocks][column block][half of the line]
    auto load_codes = [&](int c, int cp) __attribute__((always_inline)) {
        const uint32_t l = hidden((uint32_t)lane);
#pragma unroll
        for (int i = 0; i < 2; i++)
#pragma unroll
            for (int r = 0; r < 2; r++) {
                const uint32_t in_row = min((uint32_t)c * 128 + (l >> 3 & 1) * 64 + (l >> 4) * 16, row_bytes - 16u);
                cw[cp][i][r] = load_at<u32x4_t>(wt[second(cp * 2)], __umul24(row(cp * 2 + i, (int)(l & 7) + 8 * r), row_bytes) + in_row);
            }
    };
    auto in_order = [&](int cp) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < 2; i++)
#pragma unroll
            for (int k = 0; k < 4; k++) {
                const int lo = (int)cw[cp][i][0][k], hi = (int)cw[cp][i][1][k];
                cw[cp][i][0][k] = (uint32_t)__builtin_amdgcn_update_dpp(lo, hi, 0x128, 0xf, 0xc, false);  // row_ror 8, lanes 8..15
                cw[cp][i][1][k] = (uint32_t)__builtin_amdgcn_update_dpp(hi, lo, 0x128, 0xf, 0x3, false);  // lanes 0..7
            }
    };
    // Scales (or biases) 16 seg + 4 q .. + 3 of the row of lane (n, q).  Loads stay inside the row; in_segment() brings to the front what
    // was asked for, zeros behind the end of K.  (Apart, or the load would be waited for where it is issued.)
    auto load_sb = [&](const global_t (&base)[2], int seg, int cp, uint32_t (&to)[2][2]) __attribute__((always_inline)) {
        const int l = (int)hidden((uint32_t)lane);
#pragma unroll
        for (int i = 0; i < 2; i++) {
            const uint32_t e = (uint32_t)min(seg * kElements + (l >> 4) * 4, groups - 4);
            const u32x2_at2_t v = load_at<u32x2_at2_t>(base[second(cp * 2)], __umul24(row(cp * 2 + i, l & 15), sb_bytes) + e * 2);
            to[i][0] = v[0], to[i][1] = v[1];
        }
    };
    auto in_segment = [&](int seg, uint32_t (&v)[2][2]) __attribute__((always_inline)) {
        if ((seg + 1) * kElements <= groups) return;
        const int past = seg * kElements + (int)(hidden((uint32_t)lane) >> 4) * 4 - (groups - 4);  // elements in front of what was asked for
#pragma unroll
        for (int i = 0; i < 2; i++) {
            uint64_t u = (uint64_t)v[i][1] << 32 | v[i][0];
            u = past > 3 ? 0 : u >> (past > 0 ? past * 16 : 0);
            v[i][0] = (uint32_t)u, v[i][1] = (uint32_t)(u >> 32);
        }
    };
    auto meet = [&]() __attribute__((always_inline)) {
        // (bare: __syncthreads() would wait for the loads in flight)
        __builtin_amdgcn_sched_barrier(0);
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
    };
    // Everything the tile starts with is on its way before anything is waited for (one load after the other, with a list of routes,
    // a scan of scales and a first piece of x that each wait for the one before, a tile of three steps took 33 us, 1408 of them 66).
    constexpr int BATCH = 4;  // segments of scales asked for together
    load_codes(0, 0);
    load_codes(0, 1);
    uint32_t sv[BATCH][2][2][2];
    uint32_t sc[2][2][2], bi[2][2];  // scales and biases of the segment
    auto load_batch = [&](int seg0) __attribute__((always_inline)) {
#pragma unroll
        for (int s = 0; s < BATCH; s++)
            if (s == 0 || seg0 + s < segments) {
#pragma unroll
                for (int cp = 0; cp < 2; cp++) load_sb(st, seg0 + s, cp, sv[s][cp]);
            }
    };
    load_batch(0);
    __builtin_amdgcn_sched_barrier(0);
    if (tid < kRouteRows) {
        route[tid] = my_route;
        x_at[tid] = (uint32_t)my_x * (uint32_t)(steps * kStep * 2);
        sum_at[tid] = (uint32_t)my_x * (uint32_t)(segments * kElements * 4);
    }
    meet();
    const float my_down = a.rs[my_x];

    // the power of two that brings a row's largest scale into [2^10, 2^11)
#pragma unroll
    for (int i = 0; i < 8; i++) sc[i >> 2][i >> 1 & 1][i & 1] = sv[0][i >> 2][i >> 1 & 1][i & 1];
    uint32_t mag[4] = {0u, 0u, 0u, 0u};
    for (int seg0 = 0;;) {
#pragma unroll
        for (int s = 0; s < BATCH; s++)
            if (seg0 + s < segments) {
#pragma unroll
                for (int cp = 0; cp < 2; cp++) {
                    in_segment(seg0 + s, sv[s][cp]);
#pragma unroll
                    for (int i = 0; i < 2; i++) mag[cp * 2 + i] = most_of(most_of(mag[cp * 2 + i], sv[s][cp][i][0]), sv[s][cp][i][1]);
                }
            }
        seg0 += BATCH;
        if (seg0 >= segments) break;
        load_batch(seg0);
    }
    uint32_t up = 0;  // its biased exponents, a byte for each column block
#pragma unroll
    for (int cg = 0; cg < 4; cg++) {
        up |= (uint32_t)(127 + exponent_shift(max_lanes<16>(mag[cg]), 10)) << (8 * cg);
    }
    auto col_up = [&](int cg) { return __uint_as_float((hidden(up) >> (8 * cg) & 0xffu) << 23); };
    const uint32_t mask_s = opaque_s(0x03C003C0u), magic_v = opaque_v(0x4C004C00u);
    const uint32_t get_at = (uint32_t)(n * (kStep * 2) + ((q * 4 ^ n) * 16));
    const uint32_t stage_at = __builtin_amdgcn_readfirstlane(lds_offset(stage)), sums_at = __builtin_amdgcn_readfirstlane(lds_offset(sums));

    // The loop over K of a tile of RB blocks of 16 rows; its sums go to LDS, [wavefront][row][column of the wavefront].
    auto tile = [&](auto rb_tag) __attribute__((always_inline)) {
        constexpr int RB = decltype(rb_tag)::value;
        // x: a copy instruction of a wavefront brings the 512 bytes a step takes of each of two rows into LDS.  The sixteen 16-byte places of
        // a half of a row are turned against those of its neighbours (what a lane fetches, not where it lands), so that one place of
        // sixteen rows is read from all banks.
        auto copy_x = [&](int c, int to) __attribute__((always_inline)) {
            // (offsets from LDS each time: registers are short)
            const uint32_t l = hidden((uint32_t)lane), r = (uint32_t)(wave * 2) + l / 32;
            uint32_t off[2 * RB];
#pragma unroll
            for (int i = 0; i < 2 * RB; i++) off[i] = x_at[r + i * kWaves * 2];
#pragma unroll
            for (int i = 0; i < 2 * RB; i++)
                copy16_to_lds(reinterpret_cast<const uint8_t*>(a.xf) + c * (kStep * 2), off[i] + ((l & 31) ^ (r + i * kWaves * 2 & 15)) * 16u,
                              stage_at + (uint32_t)(to * RB * kStage + (i * kWaves + wave) * 1024));
        };
        copy_x(0, 0);
        f32x4_t acc[RB][4];
#pragma unroll
        for (int rb = 0; rb < RB; rb++)
#pragma unroll
            for (int cg = 0; cg < 4; cg++) acc[rb][cg] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
        if (tid < kRouteRows) down[tid] = my_down;
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // the first copies have landed
        meet();

        // The sums of x of a segment go through LDS too, a copy instruction for a block of 16 rows: lane (n, q) finds those of the
        // groups whose scales it holds where its lane's copy has put them.
        auto copy_sums = [&](int seg) __attribute__((always_inline)) {
            if (wave >= RB) return;
            const uint32_t l = hidden((uint32_t)lane);
            copy16_to_lds(a.xs, sum_at[wave * 16 + (l & 15)] + ((uint32_t)(seg * kElements) + (l >> 4) * 4) * 4, sums_at + (uint32_t)wave * 1024);
        };
        // bias and 8 * scale times the sums of x over the segment (two bf16 a sum: two slots of a product for either).  The two nearly cancel,
        // so a product takes both of eight groups.  (All biases in one and all scales in the next left the accumulator with the large half
        // in between.  fp32 error against float64, tiles of 32 routes / so / here: groups of 64, K of 704 1.69e-7 / 1.84e-7 / 1.63e-7, of
        // 4096 4.04e-7 / 4.15e-7 / 4.02e-7, of 32, K of 576 1.70e-7 / 1.82e-7 / 1.53e-7, of 128, K of 1280 2.24e-7 / 2.35e-7 / 2.17e-7; 173 us the block both ways.)
        auto affine = [&](int cp) __attribute__((always_inline)) {
#pragma unroll
            for (int i = 0; i < 2; i++) {
                const int cg = cp * 2 + i;
                uint32_t bw[4], ew[4];
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    const uint32_t sv = e & 1 ? sc[cp][i][e / 2] & 0xffff0000u : sc[cp][i][e / 2] << 16;
                    const uint32_t bv = e & 1 ? bi[i][e / 2] & 0xffff0000u : bi[i][e / 2] << 16;
                    bw[e] = dup16(__float_as_uint(__uint_as_float(bv) * col_up(cg)) >> 16);
                    ew[e] = dup16(__float_as_uint(__uint_as_float(sv) * col_up(cg) * 8.0f) >> 16);
                }
#pragma unroll
                for (int rb = 0; rb < RB; rb++) {
                    const uint4 x4 = *reinterpret_cast<const uint4*>(sums + rb * 256 + lane * 4);
                    acc[rb][cg] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, make_uint4(x4.x, x4.x, x4.y, x4.y)),
                                                                          __builtin_bit_cast(bf16x8_t, make_uint4(bw[0], ew[0], bw[1], ew[1])), acc[rb][cg], 0, 0, 0);
                    acc[rb][cg] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, make_uint4(x4.z, x4.z, x4.w, x4.w)),
                                                                          __builtin_bit_cast(bf16x8_t, make_uint4(bw[2], ew[2], bw[3], ew[3])), acc[rb][cg], 0, 0, 0);
                }
            }
        };

        // Step c, U = c % 2.  x lies in stage U; the next step's is copied into the other, whose readers have passed the barrier that ended the
        // step before, and a pair of column blocks asks for its next codes once it has used these.  The compiler, which cannot count the
        // copies, waits at a first use of codes until no more than the loads behind them are on their way, copies among them.
        // (Past the end of K the last codes and scales are asked for again: where loads may or may not have gone out the compiler counts the
        // fewest, and waited for all codes at each first use; a last step of its own cost 4 us a tile, its instructions come from memory.)
        auto step = [&](auto u_tag, int c) __attribute__((always_inline)) {
            constexpr int U = decltype(u_tag)::value;
            const bool more = c + 1 < steps;
            const int seg = c / SPS, in_seg = c % SPS;
            const bool ends = !more || in_seg == SPS - 1;  // the segment does
            const bool whole = c * 2 + 1 < pieces;  // K does not end in the step's first half
            // A's fragments of a word are read over those just multiplied, while the next word of codes is expanded; a half's scales (of
            // element e of the segment, from lane e / 4) are asked for ahead of the half before it.
            f16x8_t af[RB];
            auto read_a = [&](int half, int T, int rb) __attribute__((always_inline)) {
                const uint8_t* const at = stage + (hidden(get_at) ^ (uint32_t)(T * 16)) + U * RB * kStage + half * 256;
                af[rb] = *reinterpret_cast<const f16x8_t*>(at + rb * kStage);
            };
            uint32_t raw[2];
            auto ask_scales = [&](int cp, int half) __attribute__((always_inline)) {
                const int from = (int)(hidden((uint32_t)lane) & 15) * 4 + (GRP == 32 ? U * 2 + half : GRP == 64 ? in_seg : in_seg / 2) * 64;
#pragma unroll
                for (int i = 0; i < 2; i++) {
                    raw[i] = (uint32_t)__builtin_amdgcn_ds_bpermute(from, (int)sc[cp][i][GRP == 32 ? 0 : GRP == 64 ? half : U]);
                    if constexpr (GRP == 32) {
                        const uint32_t other = (uint32_t)__builtin_amdgcn_ds_bpermute(from, (int)sc[cp][i][1]);
                        raw[i] = q & 2 ? other : raw[i];
                    }
                }
            };
#pragma unroll
            for (int rb = 0; rb < RB; rb++) read_a(0, 0, rb);
            if (ends) load_sb(bt, seg, 0, bi);
#pragma unroll
            for (int cp = 0; cp < 2; cp++) {
                if (U == 0 && in_seg == 0) in_segment(seg, sc[cp]);
                ask_scales(cp, 0);
                in_order(cp);
                if (cp == 0) {
                    if (more) copy_x(c + 1, U ^ 1);
                    if (U == 0 && in_seg == 0) copy_sums(seg);
                }
#pragma unroll
                for (int half = 0; half < 2; half++) {
                    if (half == 1 && !whole) continue;
                    f16x2_t s2[2], m24[2];
#pragma unroll
                    for (int i = 0; i < 2; i++) {
                        const bool high = GRP == 32 ? (q & 1) != 0 : GRP == 64 ? q >= 2 : half == 1;
                        const float sv = __uint_as_float(high ? raw[i] & 0xffff0000u : raw[i] << 16) * col_up(cp * 2 + i), mv = sv * -24.0f;
                        s2[i] = f16x2_t{(_Float16)sv, (_Float16)sv};
                        m24[i] = f16x2_t{(_Float16)mv, (_Float16)mv};
                    }
                    if (half == 0) ask_scales(cp, 1);
#pragma unroll
                    for (int T = 0; T < 4; T++) {
                        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                        for (int i = 0; i < 2; i++) {
                            const uint32_t w = cw[cp][i][half][T];
                            // the pairs of a word in order: (c0, c4)(c1, c5)(c2, c6)(c3, c7), as scale * (16 + code) - 24 * scale
                            auto two = [&](uint32_t at) {
                                return __builtin_bit_cast(uint32_t, __builtin_elementwise_fma(__builtin_bit_cast(f16x2_t, and_or(at, mask_s, magic_v)), s2[i], m24[i]));
                            };
                            const f16x8_t bf = __builtin_bit_cast(f16x8_t, make_uint4(two(w << 6), two(w << 2), two(w >> 2), two(w >> 6)));
#pragma unroll
                            for (int rb = 0; rb < RB; rb++) {
                                acc[rb][cp * 2 + i] = __builtin_amdgcn_mfma_f32_16x16x32_f16(af[rb], bf, acc[rb][cp * 2 + i], 0, 0, 0);
                                if (i == 1 && !(cp == 1 && half == 1 && T == 3)) read_a(T < 3 ? half : half == 0 && whole ? 1 : 0, (T + 1) & 3, rb);
                            }
                        }
                    }
                    __builtin_amdgcn_sched_barrier(0);
                }
                if (ends) {
                    if (cp == 0 && in_seg == 0) {  // (its sums went out in this step)
                        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
                        meet();
                    }
                    in_segment(seg, bi);
                    affine(cp);
                    load_sb(st, min(seg + 1, segments - 1), cp, sc[cp]);
                }
                if (ends && cp == 0) load_sb(bt, seg, 1, bi);
                load_codes(min(c + 1, steps - 1), cp);
            }
            // x of the next step has landed: its copies went out ahead of all its codes
            asm volatile("s_waitcnt vmcnt(8)" ::: "memory");
            meet();
        };
        // A SIMD issues for its oldest wavefront first, so that the tiles of a CU would end one after the other, the last one alone and
        // waiting for itself: who is behind goes first instead.
        __builtin_amdgcn_s_setprio(3);
        for (int c = 0;;) {
            step(std::integral_constant<int, 0>{}, c);
            if (++c == steps) break;
            if (c * 4 > steps * 3)
                __builtin_amdgcn_s_setprio(0);
            else if (c * 2 > steps)
                __builtin_amdgcn_s_setprio(1);
            else if (c * 4 > steps)
                __builtin_amdgcn_s_setprio(2);
            step(std::integral_constant<int, 1>{}, c);
            if (++c == steps) break;
        }
        // (every read of the stages has returned, and every copy has landed)
        float* const mine = reinterpret_cast<float*>(stage) + wave * (kRouteRows * 64) + n;
#pragma unroll
        for (int rb = 0; rb < RB; rb++)
#pragma unroll
            for (int r = 0; r < 4; r++)
#pragma unroll
                for (int cg = 0; cg < 4; cg++) mine[(rb * 16 + 4 * q + r) * 64 + cg * 16] = acc[rb][cg][r] * (1.0f / col_up(cg));
    };
    if (count <= 16)
        tile(std::integral_constant<int, 1>{});
    else if (count <= 32)
        tile(std::integral_constant<int, 2>{});
    else
        tile(std::integral_constant<int, 3>{});

    // The row's power of two comes off, the gate's activation goes on, and the rows leave in pieces of eight columns.  (One copy of this
    // code for every number of row blocks, a piece at a time: unrolled over the tile it went past what the instruction cache holds.)
    __syncthreads();
    const float* const tile_at = reinterpret_cast<const float*>(stage) + wave * (kRouteRows * 64);
    const int lanes = pair ? 4 : 8;  // that share a row
    const int c8 = lane % lanes * 8, col = n0 + wave * (pair ? 32 : 64) + c8;
    const bool wide = (reinterpret_cast<uintptr_t>(a.y) & 15) == 0 && (a.out_f32 ? (N & 3) == 0 : (N & 7) == 0) && col + 8 <= N;
#pragma nounroll
    for (int r = lane / lanes; r < count && col < N; r += kWave / lanes) {
        float v[8];
        const int to = route[r];
        const float scale = down[r];
        const float* const from = tile_at + r * 64 + c8;
#pragma unroll
        for (int e = 0; e < 8; e++) v[e] = from[e] * scale;
        if (pair) {
#pragma unroll
            for (int e = 0; e < 8; e++) v[e] = fmul_unfused(act_value(a.act, v[e]), from[32 + e] * scale);
        }
#pragma unroll
        for (int e = 0; e < 8; e++) v[e] = to < 0 ? 0.0f : v[e];  // an expert id or a row of x out of range
        const int64_t o = (int64_t)(to & INT32_MAX) * N + col;
        if (wide) {
            if (a.out_f32) {
                float4* const dst = reinterpret_cast<float4*>(static_cast<float*>(a.y) + o);
                dst[0] = make_float4(v[0], v[1], v[2], v[3]);
                dst[1] = make_float4(v[4], v[5], v[6], v[7]);
            } else {
                *reinterpret_cast<uint4*>(static_cast<uint16_t*>(a.y) + o) =
                    make_uint4(pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3]), pack_bf16x2(v[4], v[5]), pack_bf16x2(v[6], v[7]));
            }
        } else {
#pragma unroll
            for (int e = 0; e < 8; e++) {
                if (col + e >= N) continue;
                if (a.out_f32)
                    static_cast<float*>(a.y)[o + e] = v[e];
                else
                    static_cast<uint16_t*>(a.y)[o + e] = f32_to_bf16_bits(v[e]);
            }
        }
    }
}

// ---- host side ------------------------------------------------------------------------------------------------------

static size_t up256(size_t n) { return (n + 255) & ~(size_t)255; }
static size_t fragment_bytes(int rows, int K) { return up256((size_t)rows * ((K + kStep - 1) / kStep * kStep) * 2); }
static size_t sum_bytes(int rows, int K, int group_size) { return up256((size_t)rows * ((K / group_size + kElements - 1) / kElements * kElements) * 4); }

int qmmr_strips(int N, bool pair) {
    const int cols = pair ? kCols / 2 : kCols;
    return (N + cols - 1) / cols;
}

bool qmmr_fits(int rows, int K, int N, int group_size, int bits) {
    // (32-bit offsets into the copy of x and into a tile's weight rows)
    return bits == 4 && (group_size == 32 || group_size == 64 || group_size == 128) && K % 64 == 0 && K % group_size == 0 && K >= 4 * group_size && K >= 128 && N > 0 &&
           fragment_bytes(rows, K) < ((size_t)1 << 31) && (int64_t)K * kCols < ((int64_t)1 << 31);
}

size_t qmmr_workspace_bytes(int rows, int K, int group_size) {
    return fragment_bytes(rows, K) + sum_bytes(rows, K, group_size) + up256((size_t)rows * 4);
}

hipError_t qmmr_launch(const QmmRouteCall& c, void* workspace, hipStream_t stream) {
    if (!qmmr_fits(c.rows, c.K, c.N, c.group_size, 4)) return hipErrorInvalidValue;
    QmmRouteArgs a{};
    char* p = static_cast<char*>(workspace);
    uint16_t* const xf = reinterpret_cast<uint16_t*>(p);
    uint32_t* const xs = reinterpret_cast<uint32_t*>(p += fragment_bytes(c.rows, c.K));
    float* const rs = reinterpret_cast<float*>(p += sum_bytes(c.rows, c.K, c.group_size));
    const size_t list_lds = group_staged_bytes(c.lists);
    const int first = list_lds <= kListLds ? 1 : 0;
    if (!first)
        if (hipError_t rc = moe_group_launch(c.lists, stream)) return rc;
    const auto prep = c.group_size == 32 ? qmmr_prep_kernel<32> : c.group_size == 64 ? qmmr_prep_kernel<64> : qmmr_prep_kernel<128>;
    hipLaunchKernelGGL(prep, dim3((unsigned)(first + (c.rows + kPrepThreads / kWave - 1) / (kPrepThreads / kWave))), dim3(kPrepThreads), first ? list_lds : 0,
                       stream, c.x, xf, xs, rs, c.rows, c.K, c.by_route ? c.lists.lhs : nullptr, c.lists.x_rows, c.lists, first);
    if (hipError_t rc = hipGetLastError()) return rc;
    a.xf = xf;
    a.xs = xs;
    a.rs = rs;
    a.w = c.w;
    a.s = c.s;
    a.b = c.b;
    a.y = c.y;
    a.K = c.K;
    a.N = c.N;
    a.pair = c.pair;
    a.act = c.act;
    a.out_f32 = c.out_f32;
    a.by_route = c.by_route;
    a.expert_rows = c.expert_rows;
    a.row_base = c.row_base;
    a.row_base2 = c.row_base2;
    a.chunks = c.lists.chunks;
    a.route_x = c.lists.route_x;
    a.route_of = c.lists.route_of;
    a.strips = qmmr_strips(c.N, c.pair != 0);
    const auto fn = c.group_size == 32 ? qmmr_kernel<32> : c.group_size == 64 ? qmmr_kernel<64> : qmmr_kernel<128>;
    a.most_chunks = c.lists.most_chunks;
    hipLaunchKernelGGL(fn, dim3((unsigned)((c.lists.most_chunks + 7) / 8 * 8 * a.strips)), dim3(kThreads), 0, stream, a);
    return hipGetLastError();
}

}  // namespace aq
