// affine_qmv for 2..64 rows of x on gfx950 (batched / speculative-verify decode), 4- and 8-bit codes in
// groups of 32, 64 and 128: the weights streamed exactly once (twice from 33 rows of x on), no pass over x beforehand; one launch,
// and one that adds partial tiles where the workgroups share K out.
//
// Same contract as the other matvec kernels: replaces rocm_mlx_q4_projection_batch*
// (go/engine/hip/kernels/quant/affine_projection_tuned.hipinc:292-472, 16 rows x 16 tokens in one launch) and the
// rows kernel of go/engine/metal/qmv_rows.go:14-60; semantics of MLX affine_qmv with M rows
// (go/engine/metal/kernels/quant/lthn_qmv_rows.metal:1-22).
#pragma once
#include "aq_device.h"
#include "aq_kernels.h"

#include <type_traits>

namespace aq {

namespace {

typedef const __attribute__((address_space(1))) char* gptr_t;
__device__ __forceinline__ gptr_t uniform_ptr(const void* p) {
    const uint64_t u = reinterpret_cast<uint64_t>(p);
    const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)u);
    const uint32_t hi = __builtin_amdgcn_readfirstlane((uint32_t)(u >> 32));
    return reinterpret_cast<gptr_t>(((uint64_t)hi << 32) | lo);
}
typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));
__device__ __forceinline__ uint4 load_u128_at(gptr_t base, uint32_t off) {
    const u32x4_t v = *reinterpret_cast<const __attribute__((address_space(1))) u32x4_t*>(base + off);
    return make_uint4(v[0], v[1], v[2], v[3]);
}
// The same with the non-temporal hint, for the weights: they are read once, in whole 128-byte lines per instruction, and
// leave the L1 to x, scales and biases (4096 x 14336, 16 / 32 rows of x: 12.65 -> 12.28 / 17.14 -> 16.8 us).
__device__ __forceinline__ uint4 load_u128_stream_at(gptr_t base, uint32_t off) {
    const u32x4_t v = __builtin_nontemporal_load(reinterpret_cast<const __attribute__((address_space(1))) u32x4_t*>(base + off));
    return make_uint4(v[0], v[1], v[2], v[3]);
}
__device__ __forceinline__ bf16x8_t as_bf16x8(uint32_t a, uint32_t b, uint32_t c, uint32_t d) {
    const uint4 v = make_uint4(a, b, c, d);
    return __builtin_bit_cast(bf16x8_t, v);
}

constexpr int kTokMax = 64;   // activation rows per launch (the M side), 32 per workgroup
constexpr int kTokMaxK = 16384;
constexpr int kTokWaves = 8;  // wavefronts of a workgroup, which share K
constexpr int kTokShares = 16;  // most shares of K
constexpr int kTokInsideSets = 4;  // most sets of rows of a workgroup that works through shares by itself (eight, with two sets of tokens, spill)
typedef uint32_t __attribute__((ext_vector_type(4), aligned(2))) u32x4_a2_t;  // loads of any alignment
typedef uint32_t __attribute__((ext_vector_type(2), aligned(2))) u32x2_a2_t;

}  // namespace

// v_mfma_f32_16x16x32_bf16 with 16 tokens as the rows of A (TS such sets per expanded weight: up to 16 TS rows of x) and
// 16 weight rows as the columns of B.  A workgroup of eight wavefronts owns RS sets of 16 weight rows; wavefront w takes
// the runs of 256 codes w, w + 8, ... of all of them, one run a pass.
//   * A load instruction covers whole 128-byte lines of 8 rows.  4 bit: the lines go through LDS (a wavefront's own 2.3 KiB), out
//     of which lane (n = lane % 16, q = lane / 16) reads the codes 8 q .. 8 q + 7 of row n for every step of 32 codes.  (Moves and
//     swaps between lanes instead took 125 clocks of the vector unit per set and run.)  8 bit: two DPP moves per register pair
//     give lane (n, q) the codes 16 q .. 16 q + 15 of a block of 64 of row n, whose halves are its operands of the block's two
//     steps, x being loaded to match; groups of 32, where a step is a group, swap 32-lane halves besides.
//   * x is read a whole 128-byte line of each of 8 tokens per instruction: lanes i = lane % 16 < 8 take the first 64
//     bytes of token i (an even step), lanes i >= 8 the second 64 bytes of token i - 8 (the odd step behind it); a
//     second instruction does the same for tokens 8..15, and two DPP moves per register pair put the halves where the
//     A operands want them.  Inside the 16 bytes the values are permuted into the order the expansion leaves the codes
//     in.  Every wavefront reads just the runs it multiplies.  (Requests are what this kernel pays for at the L1: with
//     64 bytes of 16 tokens per instruction, and every wavefront fetching its own 8 bytes of each row's scales and
//     biases, x and the scales each cost as much time as the weights.)
//   * scales and biases of the workgroup's rows are fetched once, by all threads together, and handed round in LDS: a thread
//     takes those of one run of one row, with loads of any alignment.
//   * a quantisation group's steps end with acc += scale * D, four FMAs per lane and set of rows.
//   * the affine term is one MFMA (groups of 32: two) per run and set of rows: lane block q carries group q of the run, A = the
//     three-way bf16 split of the group's sum of x (and kLacks times it), B = (b b b s s s 0 0); the sums of x are products
//     with ones, which leave them in every lane of their token.
//   * a wavefront keeps the A operands of its run in registers and streams the sets of rows past them, RING sets in
//     flight (see the loop); the wavefronts' partial sums meet in LDS.
// Token t of an M-row call equals token t of any other call with the same shares of K (qmvt_split), bit for bit.
// Any K that is a multiple of 64: a run that K ends inside reads its last 16 bytes again and multiplies them with zeros of x
// under scales of zero.
// What the operand holds of a code, and why.  A weight is near zero on average: what the operand has beside it comes off again,
// in the affine term, out of a sum many times the result.  Errors against the float64 product (fp32 results, relative): 4 bit,
// 128 + code 1.8-2.1e-6, 16 + code 2.8e-7, the code 1.3e-7; groups of 32 start a group's sum at -8 times its sum of x (read back
// from LDS as the C operand), which makes it the code - 8: 1.0e-7, as (code - 8) / 16 in the operand gives, for 7 vector
// instructions a word of eight codes instead of 14 (unpack4_codes).  8 bit: code - 128 0.9-1.0e-7, the code 1.4e-7.
// Measured (us, graph replay over 640 MB of weights; moves between lanes, 14 or 8 instructions a word and at most 64 rows a
// workgroup -> here): 21 rows of x, groups of 32: 3840 x (15360 | 15360) 49.5 -> 30.7, 15360 x 3840 29.6 -> 21.9; groups of 64:
// 16 / 32 rows of 4096 x 14336 12.3 -> 11.7 / 17.2 -> 16.7, 32 of 14336 x 4096 30.8 -> 19.1, 8 bit 33.9 -> 22.5.
// Bound by waits: 32 rows of 4096 x 14336 in groups of 64 take 10 us beside the 6 to 7 us of any call (launch, the first requests, the
// sums over wavefronts, the store); by counters 5 of those are vector issue and 2 matrix cores, wavefronts stand at a counter or barrier
// 35 % of their cycles (groups of 32, 21 rows of 3840 x (15360 | 15360): 53 %, vector issue 30 % of SIMD cycles, matrix cores 11 %).
// Dense groups of 32 also test every sum for infinities, which the any-width kernel keeps (plain_dot_g32).
// PAIR: the first half of the workgroup's sets of rows belongs to the gate matrix, the second half to the same rows of the
// up matrix, and the store is act(gate) * up: one pass over x and one launch for a gated MLP's two projections.
// GROUPED (expert slabs): the rows of x of a launch are the routes of one chunk of the list a.chunks (aq_moe_group.hip):
// up to 16 TS routes that name the same expert, which then streams its weights once for all of them.
// a.ksplit > 1: the workgroups of a band of rows share K out, a.share runs each, and store fp32 partial tiles [ksplit][M][N]
// ([ksplit][M][gate N | up N] for a pair) that tok_reduce_kernel adds in order.  a.inside > 1 (INSIDE): a workgroup works through
// that many shares by itself and adds their sums in the same order.
constexpr int kTokRowPitch = 144;  // LDS bytes between the 128-byte lines of a wavefront's rows: reads of 4 q + 16 step fall into different banks
// LDS bytes of the staged scales and biases of `rows` weight rows over `runs` runs, 16-byte pieces at an odd pitch so that the 16
// rows a wavefront reads at once fall into different banks
__host__ __device__ constexpr int tok_sb_pitch(bool g32, int runs) { return g32 ? 2 * runs + 1 : runs | 1; }
__host__ __device__ constexpr size_t tok_sb_bytes(bool g32, int rows, int runs) { return (size_t)rows * tok_sb_pitch(g32, runs) * 16; }
// ... of a wavefront's lines of weights (4 bit), and its sums of x where a group's sum starts from them
__host__ __device__ constexpr int tok_line_bytes(int bits) { return bits == 4 ? 16 * kTokRowPitch : 0; }
__host__ __device__ constexpr bool tok_from_sum(int bits, bool g32) { return bits == 4 && g32; }
__host__ __device__ constexpr int tok_own_bytes(int bits, bool g32, int ts) { return tok_line_bytes(bits) + (tok_from_sum(bits, g32) ? ts * 512 : 0); }

template <int BITS, int RS, int RING, int TS, int GRP, bool PAIR, bool GROUPED, bool INSIDE = false>
__device__ __forceinline__ void qmv_tok16_body(const TokArgs& a, const int block_of_all) {
    static_assert(BITS == 4 || BITS == 8, "code width");
    static_assert(GRP == 64 || GRP == 32, "group size (64: and 128)");
    constexpr int NW = kTokWaves;
    constexpr bool G32 = GRP == 32;
    constexpr int GPR = 256 / GRP;  // groups of a run (groups of 128: two, each held twice)
    constexpr bool FROM_SUM = tok_from_sum(BITS, G32);
    constexpr float kLacks = BITS == 8 ? 128.0f : G32 ? 8.0f : 0.0f;  // in codes
    static_assert(!PAIR || RS % 2 == 0, "a pair shares its sets of rows between two matrices");
    constexpr int PAIRS = PAIR ? 2 : 1;
    constexpr int LINES = BITS / 4;  // 128-byte lines of a row per run of 256 codes
    extern __shared__ __attribute__((aligned(16))) unsigned char lds_raw[];
    constexpr int ROWS = RS * 16;   // weight rows per workgroup
    constexpr int OUTS = ROWS / PAIRS;  // of each matrix
    constexpr int NT = NW * kWave;
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int n = lane & 15;
    const int q = lane >> 4;
    const int K = a.K, N = a.N;
    int block = block_of_all, split = 0, M = a.M, m0 = 0;
    if constexpr (!GROUPED) {
        const int bands = (N + OUTS - 1) / OUTS;
        if (__builtin_expect(M > a.tokens, 0)) {
            // more rows of x than a workgroup takes: eight bands for the first of them, then the same eight for the next, so that
            // the workgroups of a band run side by side on one XCD (every eighth workgroup) and share its weights in L2
            const int parts = (M + a.tokens - 1) / a.tokens, round = block / (8 * parts), in = block - round * 8 * parts;
            m0 = in / 8 * a.tokens;
            M = min(a.tokens, M - m0);
            block = round * 8 + in % 8;
            if (block >= bands * max(a.ksplit, 1)) return;
        }
        if (__builtin_expect(a.ksplit > 1, 0)) {
            split = block / bands;
            block -= split * bands;
        }
    }
    const int quads = (K + 255) >> 8;
    const int qfirst = GROUPED ? 0 : split * a.share, qend = !GROUPED && a.ksplit > 1 ? min(quads, qfirst + a.share) : quads;
    const int runs = qend - qfirst;
    const int row0 = block * OUTS;
    const uint32_t row_bytes = (uint32_t)(K * BITS / 8);
    const int groups = K >> a.gs_shift;  // of a row
    // GROUPED: this chunk's expert, its first place in the list of routes and their number
    int first_route = 0;
    size_t wrow = 0, wrow2 = 0;  // first weight row of the slab this launch reads (PAIR: of either matrix)
    uint32_t sb_end[2] = {(uint32_t)N * (uint32_t)groups, (uint32_t)N * (uint32_t)groups};  // groups from there to the end of the matrix
    if constexpr (GROUPED) {
        const RouteChunk ch = a.chunks[blockIdx.y];
        if (ch.count == 0) return;  // behind the end of the list
        M = ch.count;
        first_route = ch.first;
        wrow = (size_t)ch.expert * (size_t)a.expert_rows + (size_t)a.row_base;
        wrow2 = (size_t)ch.expert * (size_t)a.expert_rows + (size_t)a.row_base2;
        const uint64_t all = (uint64_t)a.num_experts * (uint64_t)a.expert_rows;
        sb_end[0] = (uint32_t)min((all - wrow) * (uint64_t)groups, (uint64_t)UINT32_MAX);
        if (PAIR) sb_end[1] = (uint32_t)min((all - wrow2) * (uint64_t)groups, (uint64_t)UINT32_MAX);
    }
    const size_t sb_row_bytes = (size_t)groups * 2u;
    const gptr_t wg = uniform_ptr(a.w) + wrow * row_bytes, sg = uniform_ptr(a.s) + wrow * sb_row_bytes,
                 bg = uniform_ptr(a.b) + wrow * sb_row_bytes, xg = uniform_ptr(a.x) + (size_t)m0 * K * 2;
    [[maybe_unused]] const gptr_t wg2 = PAIR ? uniform_ptr(a.w2) + wrow2 * row_bytes : wg,
                                  sg2 = PAIR ? uniform_ptr(a.s2) + wrow2 * sb_row_bytes : sg,
                                  bg2 = PAIR ? uniform_ptr(a.b2) + wrow2 * sb_row_bytes : bg;
    // weights: lane (i, q) of load `ab` reads row (i % 8) + 8 ab of a set, bytes 64 (i / 8) + 16 q of a line
    const uint32_t part16 = (uint32_t)(n >> 3) * 64u + (uint32_t)q * 16u;
    const uint32_t w_lane = (uint32_t)(row0 + (n & 7)) * row_bytes, w_last = (uint32_t)(N - 1) * row_bytes;
    // x: lane (i, q) of load `ab` of token set ts reads token 16 ts + (i % 8) + 8 ab, bytes 64 (i / 8) + 16 q of a
    // 128-byte step pair (TS sets of 16 tokens share every expanded weight); 8 bit: a step takes 8 of the 16 codes that lane
    // block q has of a block of 64, so bytes 32 q + 16 (i / 8)
    const uint32_t x_part = BITS == 4 ? part16 : (uint32_t)q * 32u + (uint32_t)(n >> 3) * 16u;
    auto x_row = [&](int t) { return GROUPED ? (uint32_t)max(a.route_x[first_route + t], 0) : (uint32_t)t; };
    uint32_t x_lane[TS][2];
#pragma unroll
    for (int ts = 0; ts < TS; ts++)
#pragma unroll
        for (int ab = 0; ab < 2; ab++) x_lane[ts][ab] = x_row(min(16 * ts + (n & 7) + 8 * ab, M - 1)) * (uint32_t)K * 2u + x_part;

    f32x4_t acc[RS][TS];
#pragma unroll
    for (int rs = 0; rs < RS; rs++)
#pragma unroll
        for (int ts = 0; ts < TS; ts++) acc[rs][ts] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};

    // Scales and biases of the workgroup's rows: the loads go out first, the first pass's x and weights behind them, and only
    // then are they stored.  Piece p: those of run p % runs of row p / runs.  What lies past the end of a row is zero; a piece
    // that would reach past the end of the matrix is read from its last bytes and moved down.
    uint4* const sbq = reinterpret_cast<uint4*>(lds_raw);
    const int sb_pitch = tok_sb_pitch(G32, runs);
    const int per = G32 ? 8 : 256 >> a.gs_shift;
    constexpr uint32_t LD = G32 ? 8 : 4;  // groups a load brings
    constexpr int PRE = 2;
    const int pieces = ROWS * runs;
    const float per_run = __builtin_amdgcn_rcpf((float)runs);
    uint4 sv[PRE], bv[PRE];
    auto piece_at = [&](int p, int& r, int& c) {
        r = (int)(((float)p + 0.5f) * per_run);  // (p / runs: p below 2^13 and runs up to 64, far from where rounding matters)
        c = p - r * runs;
        return (uint32_t)min(row0 + r % OUTS, N - 1) * (uint32_t)groups + (uint32_t)((qfirst + c) * per);
    };
    auto load_one = [&](gptr_t base, uint32_t at, uint32_t end) {
        const gptr_t from = base + min(at, end - LD) * 2u;
        if constexpr (G32) {
            const u32x4_a2_t u = *reinterpret_cast<const __attribute__((address_space(1))) u32x4_a2_t*>(from);
            return make_uint4(u[0], u[1], u[2], u[3]);
        } else {
            const u32x2_a2_t u = *reinterpret_cast<const __attribute__((address_space(1))) u32x2_a2_t*>(from);
            return make_uint4(u[0], u[1], 0u, 0u);
        }
    };
    auto load_piece = [&](int p, uint4& s, uint4& b) {
        int r, c;
        const uint32_t at = piece_at(p, r, c);
        const bool second = PAIR && r >= OUTS;
        s = load_one(second ? sg2 : sg, at, sb_end[second ? 1 : 0]);
        b = load_one(second ? bg2 : bg, at, sb_end[second ? 1 : 0]);
    };
    auto put_piece = [&](int r, int c, const uint32_t (&v)[2][4]) {
        if constexpr (G32) {
            sbq[r * sb_pitch + 2 * c] = make_uint4(v[0][0], v[0][1], v[0][2], v[0][3]);
            sbq[r * sb_pitch + 2 * c + 1] = make_uint4(v[1][0], v[1][1], v[1][2], v[1][3]);
        } else if (a.gs_shift == 7) {  // groups of 128 fill two places of 64
            sbq[r * sb_pitch + c] = make_uint4((v[0][0] & 0xffffu) * 0x10001u, (v[0][0] >> 16) * 0x10001u, (v[1][0] & 0xffffu) * 0x10001u,
                                               (v[1][0] >> 16) * 0x10001u);
        } else {
            sbq[r * sb_pitch + c] = make_uint4(v[0][0], v[0][1], v[1][0], v[1][1]);
        }
    };
    auto store_piece = [&](int p, const uint4& s, const uint4& b) {
        int r, c;
        const uint32_t at = piece_at(p, r, c), end = sb_end[PAIR && r >= OUTS ? 1 : 0];
        const int live = min(per, groups - (qfirst + c) * per);
        const int down = at > end - LD ? (int)(at - (end - LD)) : 0;
        uint32_t v[2][4] = {{s.x, s.y, s.z, s.w}, {b.x, b.y, b.z, b.w}};
        if (__builtin_expect(live != per || down != 0, 0)) {
#pragma unroll
            for (int i = 0; i < 2; i++) {
#pragma nounroll
                for (int k = 0; k < down; k++) {
                    v[i][0] = __builtin_amdgcn_alignbyte(v[i][1], v[i][0], 2);
                    v[i][1] = __builtin_amdgcn_alignbyte(v[i][2], v[i][1], 2);
                    v[i][2] = __builtin_amdgcn_alignbyte(v[i][3], v[i][2], 2);
                    v[i][3] >>= 16;
                }
#pragma unroll
                for (int e = 0; e < 4; e++) v[i][e] = 2 * e + 1 < live ? v[i][e] : 2 * e < live ? v[i][e] & 0xffffu : 0u;
            }
        }
        put_piece(r, c, v);
    };
    // A matrix of fewer groups than one load brings (up to three rows): value by value, in a place of its own, away from the code that
    // every workgroup has to fetch.
    const bool tiny = min(sb_end[0], sb_end[1]) < LD;
    auto stage_tiny = [&](int from) {
#pragma nounroll
        for (int p = from; p < pieces; p += NT) {
            int r, c;
            const uint32_t at = piece_at(p, r, c);
            const bool second = PAIR && r >= OUTS;
            uint32_t v[2][4] = {};
#pragma unroll
            for (int i = 0; i < (int)LD; i++) {
                if (i >= per || (qfirst + c) * per + i >= groups) break;
                typedef const __attribute__((address_space(1))) uint16_t* value_ptr;
                v[0][i >> 1] |= (uint32_t)*reinterpret_cast<value_ptr>((second ? sg2 : sg) + (at + i) * 2u) << (16 * (i & 1));
                v[1][i >> 1] |= (uint32_t)*reinterpret_cast<value_ptr>((second ? bg2 : bg) + (at + i) * 2u) << (16 * (i & 1));
            }
            put_piece(r, c, v);
        }
    };
    if (__builtin_expect(!tiny, 1))
#pragma unroll
    for (int i = 0; i < PRE; i++)
        if (tid + i * NT < pieces) load_piece(tid + i * NT, sv[i], bv[i]);
    __builtin_amdgcn_sched_barrier(0);

    [[maybe_unused]] unsigned char* const w_own = lds_raw + tok_sb_bytes(G32, ROWS, runs) + wave * tok_own_bytes(BITS, G32, TS);
    [[maybe_unused]] float* const sums_own = reinterpret_cast<float*>(w_own + tok_line_bytes(BITS));  // [set of tokens][step][token]

    // A pass: one run of this wavefront, its A operands in registers, and the RS sets of rows streamed
    // past them one set at a time through a ring of RING register slots.  Loads return in the order they were issued, and
    // requests that are out at the same time come back in the order the memory likes, not in the order they are needed:
    // a set is therefore requested only RING sets ahead of its use, which keeps HBM busy during the arithmetic without
    // making the first set wait for the last.  (Requesting the next pass's x and first sets from within a pass as well: 16 x 4096
    // x 14336 12.0 -> 12.5 us, 32 rows 17.9 -> 19.1.)
    uint4 ring[RING][LINES][2];
    auto issue_set = [&](auto rs_tag, int run) {
        constexpr int rs = decltype(rs_tag)::value, SL = rs % RING;
#pragma unroll
        for (int ln = 0; ln < LINES; ln++)
#pragma unroll
            for (int ab = 0; ab < 2; ab++) {
                const uint32_t row = min(w_lane + (uint32_t)(rs % (RS / PAIRS) * 16 + 8 * ab) * row_bytes, w_last);  // past N: a valid row, never stored
                const uint32_t in_row = min((uint32_t)run * (uint32_t)(128 * LINES) + (uint32_t)ln * 128u + part16, row_bytes - 16u);
                ring[SL][ln][ab] = load_u128_stream_at(PAIR && rs >= RS / 2 ? wg2 : wg, row + in_row);
            }
    };
    // (A wavefront without a run of its own takes its share of the staging and requests nothing.  When it went through the loop with
    // the first run's x and weights, unused: 9 / 24 rows of 768 x 1024 3.7 / 5.3 us against 3.3 / 4.2, 24 of 1024 x 2048 5.4
    // against 4.5, of 1536 x 2048 in groups of 32 7.2 against 6.5.  A condition around the loop's loads instead of a loop that is
    // not entered: the kernels of eight sets and two sets of tokens spill, 32 rows of 15360 x 3840 24.9 -> 50.7.)
    bool staged = false;
    auto stage = [&]() {
        int from = tid;
        asm volatile("" : "+v"(from));  // (or what the stores need is worked out ahead of the loop, before its loads are requested)
        if (__builtin_expect(tiny, 0)) {
            stage_tiny(from);
        } else {
#pragma unroll
            for (int i = 0; i < PRE; i++)
                if (from + i * NT < pieces) store_piece(from + i * NT, sv[i], bv[i]);
            for (int p = from + PRE * NT; __builtin_expect(p < pieces, 0); p += NT) {
                uint4 s, b;
                load_piece(p, s, b);
                store_piece(p, s, b);
            }
        }
        __syncthreads();
        staged = true;
    };
    // INSIDE: a.inside shares of K one after another, each with a meeting of its own, so that the sums are those of workgroups that
    // share K out.
    int share_from = 0, share_end = INSIDE && a.inside > 1 ? a.share : runs;
    float* const red = reinterpret_cast<float*>(lds_raw + a.red_at);
    [[maybe_unused]] float* const kept = red + NW * 16 * TS * ROWS;  // the sums of the shares so far
    while (true) {
        for (int at = share_from + wave; at < share_end; at += NW) {
            const int run = qfirst + at;
            uint4 xa[TS][4], xb[TS][4];
#pragma unroll
            for (int ts = 0; ts < TS; ts++)
#pragma unroll
                for (int sp = 0; sp < 4; sp++) {
                    const uint32_t in_row = run * 256 + sp * 64 < K ? (uint32_t)run * 512u + (uint32_t)sp * 128u : 0u;  // uniform
                    xa[ts][sp] = load_u128_at(xg, x_lane[ts][0] + in_row);
                    xb[ts][sp] = load_u128_at(xg, x_lane[ts][1] + in_row);
                }
            __builtin_amdgcn_sched_barrier(0);
            issue_set(std::integral_constant<int, 0>{}, run);
            if constexpr (RING > 1 && RS > 1) issue_set(std::integral_constant<int, 1>{}, run);
            __builtin_amdgcn_sched_barrier(0);
            if (!staged) stage();

            // A operands of the run, and the three-way split of the lane block's group sum of x
            if constexpr (FROM_SUM) order_wave_lds();  // (the sums of the last run have been read)
            bf16x8_t af[TS][8], a2[TS][GPR / 4];
            const uint32_t one2 = 0x3f803f80u;
            const bf16x8_t ones = as_bf16x8(one2, one2, one2, one2);
#pragma unroll
            for (int ts = 0; ts < TS; ts++) {
                if (__builtin_expect((run + 1) * 256 > K, 0)) {
#pragma unroll
                    for (int sp = 0; sp < 4; sp++)
                        if (run * 256 + sp * 64 >= K) xa[ts][sp] = xb[ts][sp] = make_uint4(0u, 0u, 0u, 0u);
                }
                f32x4_t sum[GPR];  // (every register of lane (t, q) is token t's)
                [[maybe_unused]] uint4 held = {0u, 0u, 0u, 0u};
#pragma unroll
                for (int st = 0; st < 8; st++) {
                    // even step: lanes i >= 8 take tokens 8..15 from the second load's lanes i - 8; odd step: lanes i < 8 take
                    // tokens 0..7 from the first load's lanes i + 8
                    const uint4 va = xa[ts][st >> 1], vb = xb[ts][st >> 1];
                    uint4 v;
                    if ((st & 1) == 0) {
                        v.x = __builtin_amdgcn_update_dpp(va.x, vb.x, 0x118, 0xf, 0xc, false);
                        v.y = __builtin_amdgcn_update_dpp(va.y, vb.y, 0x118, 0xf, 0xc, false);
                        v.z = __builtin_amdgcn_update_dpp(va.z, vb.z, 0x118, 0xf, 0xc, false);
                        v.w = __builtin_amdgcn_update_dpp(va.w, vb.w, 0x118, 0xf, 0xc, false);
                    } else {
                        v.x = __builtin_amdgcn_update_dpp(vb.x, va.x, 0x108, 0xf, 0x3, false);
                        v.y = __builtin_amdgcn_update_dpp(vb.y, va.y, 0x108, 0xf, 0x3, false);
                        v.z = __builtin_amdgcn_update_dpp(vb.z, va.z, 0x108, 0xf, 0x3, false);
                        v.w = __builtin_amdgcn_update_dpp(vb.w, va.w, 0x108, 0xf, 0x3, false);
                    }
                    if constexpr (BITS == 4)  // the order the expansion leaves the codes of a word in: 0 2 4 6 1 3 5 7
                        v = make_uint4(__builtin_amdgcn_perm(v.y, v.x, 0x05040100u), __builtin_amdgcn_perm(v.w, v.z, 0x05040100u),
                                       __builtin_amdgcn_perm(v.y, v.x, 0x07060302u), __builtin_amdgcn_perm(v.w, v.z, 0x07060302u));
                    if constexpr (BITS == 8 && G32) {  // (as the codes: the even step's upper lanes against the odd one's lower)
                        if ((st & 1) == 0) {
                            held = v;
                            continue;
                        }
                        const auto x = __builtin_amdgcn_permlane32_swap(held.x, v.x, false, false);
                        const auto y = __builtin_amdgcn_permlane32_swap(held.y, v.y, false, false);
                        const auto z = __builtin_amdgcn_permlane32_swap(held.z, v.z, false, false);
                        const auto w = __builtin_amdgcn_permlane32_swap(held.w, v.w, false, false);
                        af[ts][st - 1] = as_bf16x8(x[0], y[0], z[0], w[0]);
                        sum[st - 1] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ones, af[ts][st - 1], f32x4_t{0.0f, 0.0f, 0.0f, 0.0f}, 0, 0, 0);
                        v = make_uint4(x[1], y[1], z[1], w[1]);
                    }
                    af[ts][st] = as_bf16x8(v.x, v.y, v.z, v.w);
                    const int g = st / (8 / GPR);
                    const bool begins = st % (8 / GPR) == 0;
                    sum[g] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ones, af[ts][st], begins ? f32x4_t{0.0f, 0.0f, 0.0f, 0.0f} : sum[g], 0, 0, 0);
                }
#pragma unroll
                for (int g4 = 0; g4 < GPR / 4; g4++) {
                    const float X = q == 0 ? sum[4 * g4][0] : q == 1 ? sum[4 * g4 + 1][0] : q == 2 ? sum[4 * g4 + 2][0] : sum[4 * g4 + 3][0];
                    if constexpr (FROM_SUM) sums_own[(ts * 8 + 4 * g4 + q) * 16 + n] = -8.0f * X;
                    const uint32_t u0 = __float_as_uint(X) & 0xffff0000u;
                    const float r1 = X - __uint_as_float(u0);
                    const uint32_t u1 = __float_as_uint(r1) & 0xffff0000u;
                    const uint32_t u2 = __float_as_uint(r1 - __uint_as_float(u1)) & 0xffff0000u;
                    const uint32_t m0 = __float_as_uint(kLacks * __uint_as_float(u0));
                    const uint32_t m1 = __float_as_uint(kLacks * __uint_as_float(u1));
                    const uint32_t m2 = __float_as_uint(kLacks * __uint_as_float(u2));
                    a2[ts][g4] = as_bf16x8((u0 >> 16) | u1, (u2 >> 16) | m0, (m1 >> 16) | m2, 0u);
                }
            }
            // picks element q of four bf16 values in two registers, twice
            const uint32_t sel_q = 0x01000100u + 0x02020202u * (uint32_t)q;

            auto run_set = [&](auto rs_tag) {
                constexpr int rs = decltype(rs_tag)::value, SL = rs % RING;
                // scales, then biases, of the run's groups
                uint4 sbv, bbv;
                if constexpr (G32) {
                    sbv = sbq[(rs * 16 + n) * sb_pitch + 2 * at];
                    bbv = sbq[(rs * 16 + n) * sb_pitch + 2 * at + 1];
                } else {
                    sbv = sbq[(rs * 16 + n) * sb_pitch + at];
                    bbv = make_uint4(sbv.z, sbv.w, 0u, 0u);
                }
                // the codes of a line: 4 bit the words of the set's eight steps, 8 bit the two words of each of four steps
                // (8 bit, two sets of tokens, in groups of 32 or with eight sets of rows: both lines at once, so that the next set is
                // requested before the first product; us, line by line / at once: 32 rows of 4096 x 14336 in groups of 32 22.0 / 21.7, of
                // 2560 x (10240 | 10240) 24.0 / 22.2, of 14336 x 4096 22.0 / 21.2; but 32 rows of 4096 x 14336 in groups of 64 20.0 / 20.6,
                // and one set of tokens, 4 rows, 14.6 / 15.3)
                constexpr int HELD = TS == 2 && (G32 || RS == 8) ? LINES : 1;
                uint32_t ww[8 * HELD];
                auto fetch_line = [&](int ln) {
                    const int w0 = ln % HELD * 8;
                    const uint4 la = ring[SL][ln][0], lb = ring[SL][ln][1];
                    if constexpr (BITS == 4) {
                        unsigned char* const to = w_own + (n & 7) * kTokRowPitch + part16;
                        order_wave_lds();  // (the last set's words have been read)
                        *reinterpret_cast<uint4*>(to) = la;
                        *reinterpret_cast<uint4*>(to + 8 * kTokRowPitch) = lb;
                        order_wave_lds();  // the lines, and the sums above, are there for other lanes to read
                        const unsigned char* const from = w_own + n * kTokRowPitch;
#pragma unroll
                        for (int i = 0; i < 8; i++) ww[i] = *reinterpret_cast<const uint32_t*>(from + i * 16 + q * 4);
                    } else {
                        // first 64 bytes of all 16 rows (lanes i >= 8 from the second load's lanes i - 8), second 64 bytes (lanes
                        // i < 8 from the first load's lanes i + 8): as for x
                        ww[w0] = __builtin_amdgcn_update_dpp(la.x, lb.x, 0x118, 0xf, 0xc, false);
                        ww[w0 + 1] = __builtin_amdgcn_update_dpp(la.y, lb.y, 0x118, 0xf, 0xc, false);
                        ww[w0 + 2] = __builtin_amdgcn_update_dpp(la.z, lb.z, 0x118, 0xf, 0xc, false);
                        ww[w0 + 3] = __builtin_amdgcn_update_dpp(la.w, lb.w, 0x118, 0xf, 0xc, false);
                        ww[w0 + 4] = __builtin_amdgcn_update_dpp(lb.x, la.x, 0x108, 0xf, 0x3, false);
                        ww[w0 + 5] = __builtin_amdgcn_update_dpp(lb.y, la.y, 0x108, 0xf, 0x3, false);
                        ww[w0 + 6] = __builtin_amdgcn_update_dpp(lb.z, la.z, 0x108, 0xf, 0x3, false);
                        ww[w0 + 7] = __builtin_amdgcn_update_dpp(lb.w, la.w, 0x108, 0xf, 0x3, false);
                        if constexpr (G32) {  // a step is one half of a block of 64: the second 8 codes of its lanes move across
#pragma unroll
                            for (int g = 0; g < 2; g++)
#pragma unroll
                                for (int k = 0; k < 2; k++) {
                                    const auto p = __builtin_amdgcn_permlane32_swap(ww[w0 + 4 * g + k], ww[w0 + 4 * g + 2 + k], false, false);
                                    ww[w0 + 4 * g + k] = p[0];
                                    ww[w0 + 4 * g + 2 + k] = p[1];
                                }
                        }
                    }
                    if (ln == LINES - 1) {  // (into the registers that are free now)
                        __builtin_amdgcn_sched_barrier(0);
                        if constexpr (rs + RING < RS) issue_set(std::integral_constant<int, rs + RING>{}, run);
                        __builtin_amdgcn_sched_barrier(0);
                    }
                };
                f32x4_t part[TS], d[TS];
#pragma unroll
                for (int ts = 0; ts < TS; ts++) part[ts] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
                auto step = [&](auto st_tag) {
                    constexpr int st = decltype(st_tag)::value;
                    if constexpr (st % (8 * HELD / LINES) == 0)
#pragma unroll
                        for (int ln = st * LINES / 8; ln < st * LINES / 8 + HELD; ln++) fetch_line(ln);
                    uint32_t e[4];
                    if constexpr (BITS == 4) {
                        unpack4_codes(ww[st], e);
                    } else {
                        constexpr int w0 = 2 * (st % (4 * HELD));
                        unpack8_centred(ww[w0], e);
                        unpack8_centred(ww[w0 + 1], e + 2);
                    }
                    const bf16x8_t bop = as_bf16x8(e[0], e[1], e[2], e[3]);
                    constexpr int g = st / (8 / GPR);
                    constexpr bool begins = st % (8 / GPR) == 0, ends = (st + 1) % (8 / GPR) == 0;
                    const uint32_t sw = g < 2 ? sbv.x : g < 4 ? sbv.y : g < 6 ? sbv.z : sbv.w;
                    const float sc = (g & 1) ? __uint_as_float(sw & 0xffff0000u) : __uint_as_float(sw << 16);
#pragma unroll
                    for (int ts = 0; ts < TS; ts++) {
                        f32x4_t from = {0.0f, 0.0f, 0.0f, 0.0f};
                        if constexpr (FROM_SUM) from = *reinterpret_cast<const f32x4_t*>(sums_own + (ts * 8 + st) * 16 + 4 * q);
                        d[ts] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(af[ts][st], bop, begins ? from : d[ts], 0, 0, 0);
                        if (ends)
#pragma unroll
                            for (int r = 0; r < 4; r++) {
                                float v = __builtin_fmaf(sc, d[ts][r], part[ts][r]);
                                if constexpr (G32) asm volatile("" : "+v"(v));  // here, not behind all the steps: their products would be held until then
                                part[ts][r] = v;
                            }
                    }
                };
                step(std::integral_constant<int, 0>{});
                step(std::integral_constant<int, 1>{});
                step(std::integral_constant<int, 2>{});
                step(std::integral_constant<int, 3>{});
                step(std::integral_constant<int, 4>{});
                step(std::integral_constant<int, 5>{});
                step(std::integral_constant<int, 6>{});
                step(std::integral_constant<int, 7>{});
#pragma unroll
                for (int g4 = 0; g4 < GPR / 4; g4++) {
                    const uint32_t bb = __builtin_amdgcn_perm(g4 ? bbv.w : bbv.y, g4 ? bbv.z : bbv.x, sel_q);
                    const uint32_t ss = __builtin_amdgcn_perm(g4 ? sbv.w : sbv.y, g4 ? sbv.z : sbv.x, sel_q);
                    const bf16x8_t b2 = as_bf16x8(bb, __builtin_amdgcn_perm(ss, bb, 0x05040100u), ss, 0u);
#pragma unroll
                    for (int ts = 0; ts < TS; ts++)
                        part[ts] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a2[ts][g4], b2, part[ts], 0, 0, 0);
                }
#pragma unroll
                for (int ts = 0; ts < TS; ts++)
#pragma unroll
                    for (int r = 0; r < 4; r++) acc[rs][ts][r] += part[ts][r];
                __builtin_amdgcn_sched_barrier(0);
            };
            run_set(std::integral_constant<int, 0>{});
            if constexpr (RS > 1) run_set(std::integral_constant<int, 1>{});
            if constexpr (RS > 2) run_set(std::integral_constant<int, 2>{});
            if constexpr (RS > 3) run_set(std::integral_constant<int, 3>{});
            if constexpr (RS > 4) run_set(std::integral_constant<int, 4>{});
            if constexpr (RS > 5) run_set(std::integral_constant<int, 5>{});
            if constexpr (RS > 6) run_set(std::integral_constant<int, 6>{});
            if constexpr (RS > 7) run_set(std::integral_constant<int, 7>{});
            static_assert(RS <= 8 && RS % RING == 0, "sets of rows per workgroup");
        }

        if (!staged) stage();  // a wavefront without a run of its own

        // ---- the wavefronts' partial sums meet in LDS: red[wave][token][row]; thread (token, row) adds them in wave order.  Behind
        // what is staged, so that a wavefront need not wait before it puts its own there, or in its place (tok_lds_bytes) ----
        if (a.red_at == 0) __syncthreads();
        // D layout of the 16x16 MFMA: lane (n, q), register r -> token 4 q + r (of its set), weight row n
#pragma unroll
        for (int rs = 0; rs < RS; rs++)
#pragma unroll
            for (int ts = 0; ts < TS; ts++)
#pragma unroll
                for (int r = 0; r < 4; r++) red[(wave * 16 * TS + 16 * ts + 4 * q + r) * ROWS + rs * 16 + n] = acc[rs][ts][r];
        __syncthreads();
        auto total_of = [&](int t, int column) {
            float total = red[t * ROWS + column];
#pragma unroll
            for (int p = 1; p < NW; p++) total += red[(p * 16 * TS + t) * ROWS + column];
            return total;
        };
        for (int o = tid; o < min(M, 16 * TS) * OUTS; o += NT) {
            const int t = o / OUTS, rl = o - t * OUTS;
            const int row = row0 + rl;
            if (row >= N) continue;
            float total = total_of(t, rl);
            [[maybe_unused]] float up = PAIR ? total_of(t, OUTS + rl) : 0.0f;
            if constexpr (INSIDE) {
                if (share_from > 0) total = kept[o] + total;
                if (share_end < runs) {
                    kept[o] = total;
                    continue;
                }
            }
            if (!GROUPED && a.ksplit > 1) {
                float* const dst = a.tile + ((size_t)split * a.M + m0 + t) * (size_t)(PAIRS * N);
                dst[row] = total;
                if constexpr (PAIR) dst[N + row] = up;
                continue;
            }
            if constexpr (G32 && !GROUPED) {  // (dense groups of 32 keep what the any-width kernel makes of infinities)
#pragma nounroll
                for (int part = 0; part < PAIRS; part++) {
                    if (!not_finite(part ? up : total)) continue;
                    const float v = plain_dot_g32(a.x + (size_t)(m0 + t) * K, (PAIR && part ? a.w2 : a.w) + (size_t)row * (row_bytes / 4),
                                                  (PAIR && part ? a.s2 : a.s) + (size_t)row * groups, (PAIR && part ? a.b2 : a.b) + (size_t)row * groups, K, BITS);
                    if (part) up = v; else total = v;
                }
            }
            if constexpr (PAIR) total = fmul_unfused(act_value(a.act, total), up);
            size_t y_row = (size_t)(m0 + t);
            if constexpr (GROUPED) {
                const int route = a.route_of[first_route + t];
                if (route < 0) total = 0.0f;  // an expert id or a row of x out of range
                y_row = (size_t)(route & INT32_MAX);
            }
            const size_t at = y_row * N + row;
            if (a.out_f32) {
                static_cast<float*>(a.y)[at] = total;
            } else {
                static_cast<uint16_t*>(a.y)[at] = f32_to_bf16_bits(total);
            }
        }
        if (!INSIDE || share_end >= runs) break;
        share_from = share_end;
        share_end = min(runs, share_end + a.share);
#pragma unroll
        for (int rs = 0; rs < RS; rs++)
#pragma unroll
            for (int ts = 0; ts < TS; ts++) acc[rs][ts] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
        __syncthreads();  // the last share's sums have been read
    }
}

template <int BITS, int RS, int RING, int TS, int GRP, bool PAIR>
__global__ __launch_bounds__(kTokWaves* kWave) void qmv_tok16_kernel(const TokArgs a) {
    qmv_tok16_body<BITS, RS, RING, TS, GRP, PAIR, false>(a, (int)blockIdx.x);
}
template <int BITS, int RS, int RING, int TS, int GRP, bool PAIR>
__global__ __launch_bounds__(kTokWaves* kWave) void qmv_tok16_grouped_kernel(const TokArgs a) {
    qmv_tok16_body<BITS, RS, RING, TS, GRP, PAIR, true>(a, (int)blockIdx.x);
}
// up to four matrices that share x in one grid: every workgroup belongs to one of them
template <int BITS, int RS, int RING, int TS, int GRP>
__global__ __launch_bounds__(kTokWaves* kWave) void qmv_tok16_multi_kernel(const TokMultiArgs ma) {
    int i = 0, before = 0;
    while (i + 1 < ma.count && (int)blockIdx.x >= ma.block_end[i]) before = ma.block_end[i++];
    TokArgs a{ma.common};
    a.tokens = ma.tokens;
    a.w = ma.w[i];
    a.s = ma.s[i];
    a.b = ma.b[i];
    a.y = ma.y[i];
    a.N = ma.N[i];
    a.ksplit = ma.ksplit[i];
    a.share = ma.share[i];
    a.inside = ma.inside[i];
    a.tile = ma.tile[i];
    a.red_at = ma.red_at;
    qmv_tok16_body<BITS, RS, RING, TS, GRP, false, false, RS <= kTokInsideSets>(a, (int)blockIdx.x - before);
}

// ---- kernels of one code width -------------------------------------------------------------------------------------

typedef void (*QmvTokKernel)(const TokArgs);
typedef void (*QmvTokMultiKernel)(const TokMultiArgs);
struct QmvTokEntry {
    QmvVariant v;  // m = most activation rows, rows = sets of weight rows per workgroup, waves = wavefronts that share K
                   // (depth = sets of rows in flight, xmode = runs of 256 codes a wavefront holds per pass)
    QmvTokKernel fn[2];           // [groups of 32]
    QmvTokMultiKernel multi[2];
    QmvTokKernel pair[2];         // null for one set of rows per workgroup
    QmvTokKernel grouped[2][2];   // [groups of 32][pair], four sets of rows only
    const char* name[3];          // groups of 64 with K a multiple of 256; groups of 64 or 128; groups of 32
    int wg_rows;  // weight rows per workgroup
    int ts;       // sets of 16 tokens per expanded weight (1: up to 16 rows of x, 2: up to 32)
};
#define AQ_QMVT_(BITS, TAG, M, RS, RING, TS, PAIRS, GROUPED)                                                             \
    {                                                                                                                    \
        {"qmvt_b" #BITS "_m" TAG "_r" #RS "_w8_q1_d" #RING, BITS, M, RS, 8, RING, 0, 1, 6},                               \
            {qmv_tok16_kernel<BITS, RS, RING, TS, 64, false>, qmv_tok16_kernel<BITS, RS, RING, TS, 32, false>},           \
            {qmv_tok16_multi_kernel<BITS, RS, RING, TS, 64>, qmv_tok16_multi_kernel<BITS, RS, RING, TS, 32>},             \
            PAIRS(BITS, RS, RING, TS), GROUPED(BITS, RS, RING, TS),                                                       \
            {"qmvt_b" #BITS "_m" TAG "_r" #RS "_w8_q1_d" #RING, "qmvt_b" #BITS "_m" TAG "_r" #RS "_any",                   \
             "qmvt_b" #BITS "_m" TAG "_r" #RS "_s32"},                                                                    \
            16 * RS, TS                                                                                                   \
    }
#define AQ_QMVT_NOPAIR(BITS, RS, RING, TS) {nullptr, nullptr}
#define AQ_QMVT_PAIR(BITS, RS, RING, TS) {qmv_tok16_kernel<BITS, RS, RING, TS, 64, true>, qmv_tok16_kernel<BITS, RS, RING, TS, 32, true>}
#define AQ_QMVT_NOGROUP(BITS, RS, RING, TS) {{nullptr, nullptr}, {nullptr, nullptr}}
#define AQ_QMVT_GROUP(BITS, RS, RING, TS)                                                                    \
    {                                                                                                        \
        {qmv_tok16_grouped_kernel<BITS, RS, RING, TS, 64, false>, qmv_tok16_grouped_kernel<BITS, RS, RING, TS, 64, true>}, \
        {                                                                                                    \
            qmv_tok16_grouped_kernel<BITS, RS, RING, TS, 32, false>, qmv_tok16_grouped_kernel<BITS, RS, RING, TS, 32, true> \
        }                                                                                                    \
    }
#define AQ_QMVT_SET(BITS, RING8)                                                                                    \
    AQ_QMVT_(BITS, "16", 16, 8, 2, 1, AQ_QMVT_PAIR, AQ_QMVT_NOGROUP), AQ_QMVT_(BITS, "16", 16, 4, 2, 1, AQ_QMVT_PAIR, AQ_QMVT_GROUP), \
        AQ_QMVT_(BITS, "16", 16, 2, 2, 1, AQ_QMVT_PAIR, AQ_QMVT_NOGROUP),                                      \
        AQ_QMVT_(BITS, "16", 16, 1, 1, 1, AQ_QMVT_NOPAIR, AQ_QMVT_NOGROUP),                                    \
        AQ_QMVT_(BITS, "32_s2", 32, 8, RING8, 2, AQ_QMVT_PAIR, AQ_QMVT_NOGROUP),                               \
        AQ_QMVT_(BITS, "32_s2", 32, 4, 2, 2, AQ_QMVT_PAIR, AQ_QMVT_GROUP),                                     \
        AQ_QMVT_(BITS, "32_s2", 32, 2, 2, 2, AQ_QMVT_PAIR, AQ_QMVT_NOGROUP),                                   \
        AQ_QMVT_(BITS, "32_s2", 32, 1, 1, 2, AQ_QMVT_NOPAIR, AQ_QMVT_NOGROUP)

constexpr int kTokPerWidth = 8;
const QmvTokEntry* tok_entries_4();  // aq_qmv_tok.hip
const QmvTokEntry* tok_entries_8();  // aq_qmv_tok8.hip (a source of its own: compile time)

}  // namespace aq
