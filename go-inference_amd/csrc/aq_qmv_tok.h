// affine_qmv for 2..32 rows of x on gfx950 (batched / speculative-verify decode), 4- and 8-bit codes in
// groups of 32, 64 and 128: one launch, the weights streamed exactly once, no pass over x beforehand and no partial tiles
// in memory.
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
typedef uint32_t u32x2_t __attribute__((ext_vector_type(2)));
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
__device__ __forceinline__ uint2 load_u64_at(gptr_t base, uint32_t off) {
    const u32x2_t v = *reinterpret_cast<const __attribute__((address_space(1))) u32x2_t*>(base + off);
    return make_uint2(v[0], v[1]);
}
__device__ __forceinline__ bf16x8_t as_bf16x8(uint32_t a, uint32_t b, uint32_t c, uint32_t d) {
    const uint4 v = make_uint4(a, b, c, d);
    return __builtin_bit_cast(bf16x8_t, v);
}

constexpr int kTokMax = 32;   // activation rows per launch (the M side)
constexpr int kTokMaxK = 16384;
constexpr int kTokWaves = 8;  // wavefronts of a workgroup, which share K
// 8-byte pieces of scales (and of biases) a thread of the 16-token form stages at most: K up to 16384 with 16 wavefronts
__host__ __device__ constexpr int tok16_stage_pieces(int nw) { return nw >= 16 ? 4 : 8; }

}  // namespace

// v_mfma_f32_16x16x32_bf16 with 16 tokens as the rows of A (TS such sets per expanded weight: up to 16 TS rows of x) and
// 16 weight rows as the columns of B.  A workgroup of NW wavefronts owns RS sets of 16 weight rows; wavefront w takes
// the runs of 256 codes w, w + NW, ... of all of them, QW runs per pass.
//   * A load instruction covers whole 128-byte lines (a run of 256 codes) of 8 rows; two DPP moves per register pair
//     bring two such loads into the shape "lane (n = lane % 16, p = lane / 16) holds bytes 16 p .. 16 p + 15 of a
//     64-byte block of row n".  The MFMA wants from lane (n, q) the eight codes 8 q .. 8 q + 7 of a run of 32, i.e. word
//     q of four consecutive words: the four registers are transposed across the four 16-lane blocks (four lane swaps
//     per 16 bytes), after which register i of a block of 128 codes is the B operand of its step i (codes 32 i ..
//     32 i + 31), expanded with one v_and_or_b32 per pair of codes.
//   * x is read a whole 128-byte line of each of 8 tokens per instruction: lanes i = lane % 16 < 8 take the first 64
//     bytes of token i (an even step), lanes i >= 8 the second 64 bytes of token i - 8 (the odd step behind it); a
//     second instruction does the same for tokens 8..15, and two DPP moves per register pair put the halves where the
//     A operands want them.  Inside the 16 bytes the values are permuted into the order the expansion leaves the codes
//     in.  Every wavefront reads just the runs it multiplies.  (Requests are what this kernel pays for at the L1: with
//     64 bytes of 16 tokens per instruction, and every wavefront fetching its own 8 bytes of each row's scales and
//     biases, x and the scales each cost as much time as the weights.)
//   * scales and biases of the workgroup's rows are fetched once, whole rows by all threads together, and handed round
//     in LDS.
//   * two steps make a quantisation group: acc += scale * D, four FMAs per lane, group and set of rows.
//   * the affine term is one MFMA per run and set of rows: lane block q carries group q of the run, A = the three-way
//     bf16 split of the group's sum of x (and -128 times it), B = (b b b s s s 0 0); the sums of x come from v_dot2
//     per lane and a 4 x 4 transpose-add over the lane blocks, which leaves group q's total in block q.
//   * a wavefront keeps the A operands of its runs in registers and streams the sets of rows past them, RING sets in
//     flight (see the loop); the wavefronts' partial sums meet in LDS.
// Token t of an M-row call equals token t of any other call on the same variant, bit for bit.
// 8-bit codes (BITS = 8): a run of 256 codes is two lines per row, four loads per set of rows; the 64 bytes a
// 16-lane-block row holds after the DPP moves are one quantisation group, lane (n, p) has its codes 16 p .. 16 p + 15, and
// the two halves of those are the B operands of the group's two steps as they lie (no transpose: which codes share a
// step is free as long as x follows, and x is loaded to follow: lane (t, p) takes x[64 g + 16 p + 8 i ..] for step i);
// codes become bf16 by v_cvt_f32_ubyte + v_perm (exact), in their natural order; the affine term is bias * sum(x) alone.
// ANY: K any multiple of 64 and groups of GRP = 32, or of 64 / 128.  A run that K ends inside reads its last 16 bytes
// again and multiplies them with zeros of x.  Scales and biases go to LDS element by element (the rows of a workgroup are
// one flat piece of memory, read 16 bytes a lane whatever the row pitch), which costs 8 LDS writes per 16 bytes but no
// more global requests than the aligned form.  Groups of 32: one step of the MFMA is one group, so every step ends with
// its four FMAs, and the affine term is two MFMAs per run.  8-bit codes: a lane's 16 codes lie in one group, but the step
// of 32 codes that is group 0 of a block of 64 has to come from lane blocks 0 and 1 alone: a swap of 32-lane halves
// between the two steps' registers moves the second 8 codes of those lanes to lane blocks 2 and 3 (x takes the same swap).
// What the operand holds of a code, and why.  A weight is near zero on average: what 128 + code has beside it comes off again,
// in the affine term, out of sums 28 times the result.  Errors against the float64 product (fp32 results, relative; in brackets
// the kernels these shapes had before this one): 4 bit, groups of 32 2.1e-6 with 128 + code, 1.0e-7 with (code - 8) / 16 (3..4
// rows 8.3e-7, more rows 0.9e-7); groups of 64 and 128 1.8e-6, 2.8e-7 with 16 + code (5..16 rows 8.3e-7, more 1.2e-5); 8 bit
// 1.6e-7 with the code, 0.9-1.0e-7 with code - 128 (0.9-1.4e-7).  Vector instructions per word of 4-bit codes: 7, 8 for 16 +
// code, 14 for (code - 8) / 16, which is therefore only where groups of 32 need it.
// Measured (us, graph replay over 640 MB of weights; 128 + code or the plain 8-bit code -> here): 21 x 3840 x 15360 in groups of
// 32 20.4 -> 21.9 (the any-width kernel this shape had: 0.48 ms a matrix), 32 x 4096 x 14336 21.5 -> 23.0 against 16.8 for groups
// of 64: four more FMAs a lane per 32 codes; 32 x 4032 x 14336 in groups of 64 18.4 -> 18.7, 2 us over whole runs for the
// element-wise staging; 16 x 4032 x 14336 13.6 -> 13.7, 8 bit 17.6 -> 17.8; 12 x 4096 x 14336 in groups of 128 12.3 -> 12.5.
// Dense groups of 32 also test every sum for infinities, which the any-width kernel keeps (plain_dot_g32).
// PAIR: the first half of the workgroup's sets of rows belongs to the gate matrix, the second half to the same rows of the
// up matrix, and the store is act(gate) * up: one pass over x and one launch for a gated MLP's two projections.
// GROUPED (expert slabs): the rows of x of a launch are the routes of one chunk of the list a.chunks (aq_moe_group.hip):
// up to 16 TS routes that name the same expert, which then streams its weights once for all of them.
template <int BITS, int NW, int RS, int QW, int RING, int TS, bool ANY, int GRP, bool PAIR, bool GROUPED>
__device__ __forceinline__ void qmv_tok16_body(const QmvArgs& a, const int block) {
    static_assert(BITS == 4 || BITS == 8, "code width");
    static_assert(GRP == 64 || (GRP == 32 && ANY), "group size");
    constexpr bool G32 = GRP == 32;
    constexpr int GPR = 256 / GRP;  // groups of a run
    // what the operand holds of a code: 4 bit 128 + code; ANY 16 + code, in groups of 32 (code - 8) / 16; 8 bit code; ANY code - 128
    constexpr bool CENTRED = BITS == 8 ? ANY : G32;
    constexpr float kUnit = CENTRED && BITS == 4 ? 1.0f / 16 : 1.0f;
    constexpr float kLacks = CENTRED ? (BITS == 4 ? 8.0f : 128.0f) : BITS == 8 ? 0.0f : ANY ? -16.0f : -128.0f;  // in codes
    static_assert(!PAIR || RS % 2 == 0, "a pair shares its sets of rows between two matrices");
    constexpr int PAIRS = PAIR ? 2 : 1;
    constexpr int LINES = BITS / 4;  // 128-byte lines of a row per run of 256 codes
    extern __shared__ __attribute__((aligned(16))) unsigned char lds_raw[];
    constexpr int ROWS = RS * 16;   // weight rows per workgroup
    constexpr int OUTS = ROWS / PAIRS;  // of each matrix
    constexpr int TSTRIDE = ROWS;   // floats between tokens in the LDS partials
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int n = lane & 15;
    const int q = lane >> 4;
    const int K = a.K, N = a.N;
    const int groups = K >> 6;
    const int quads = ANY ? (K + 255) >> 8 : K >> 8;
    const int row0 = block * OUTS;
    const uint32_t row_bytes = (uint32_t)(K * BITS / 8);
    // GROUPED: this chunk's expert, its first place in the list of routes and their number
    int M = a.M, first_route = 0;
    size_t wrow = 0, wrow2 = 0;  // first weight row of the slab this launch reads (PAIR: of either matrix)
    if constexpr (GROUPED) {
        const RouteChunk ch = a.chunks[blockIdx.y];
        if (ch.count == 0) return;  // behind the end of the list
        M = ch.count;
        first_route = ch.first;
        wrow = (size_t)ch.expert * (size_t)a.expert_rows + (size_t)a.row_base;
        wrow2 = (size_t)ch.expert * (size_t)a.expert_rows + (size_t)a.row_base2;
    }
    const size_t sb_row_bytes = (size_t)(ANY ? K >> a.gs_shift : groups) * 2u;
    const gptr_t wg = uniform_ptr(a.w) + wrow * row_bytes, sg = uniform_ptr(a.s) + wrow * sb_row_bytes,
                 bg = uniform_ptr(a.b) + wrow * sb_row_bytes, xg = uniform_ptr(a.x);
    [[maybe_unused]] const gptr_t wg2 = PAIR ? uniform_ptr(a.w2) + wrow2 * row_bytes : wg,
                                  sg2 = PAIR ? uniform_ptr(a.s2) + wrow2 * sb_row_bytes : sg,
                                  bg2 = PAIR ? uniform_ptr(a.b2) + wrow2 * sb_row_bytes : bg;
    // weights: lane (i, q) of load `ab` reads row (i % 8) + 8 ab of a set, bytes 64 (i / 8) + 16 q of the run's 128: an
    // instruction covers whole 128-byte lines of 8 rows
    const uint32_t w_part = (uint32_t)(n >> 3) * 64u + (uint32_t)q * 16u;  // (ANY: added per run, where it is clamped to the row)
    uint32_t w_lane[RS][2];
#pragma unroll
    for (int rs = 0; rs < RS; rs++)
#pragma unroll
        for (int ab = 0; ab < 2; ab++) {
            const int row = min(row0 + rs % (RS / PAIRS) * 16 + (n & 7) + 8 * ab, N - 1);  // past N: a valid row, never stored
            w_lane[rs][ab] = (uint32_t)row * row_bytes + (ANY ? 0u : w_part);
        }
    // x: lane (i, q) of load `ab` of token set ts reads token 16 ts + (i % 8) + 8 ab, bytes 64 (i / 8) + 16 q of a
    // 128-byte step pair (TS sets of 16 tokens share every expanded weight)
    auto x_row = [&](int t) { return GROUPED ? (uint32_t)max(a.route_x[first_route + t], 0) : (uint32_t)t; };
    uint32_t x_lane[TS][2];
#pragma unroll
    for (int ts = 0; ts < TS; ts++)
#pragma unroll
        for (int ab = 0; ab < 2; ab++)
            x_lane[ts][ab] = x_row(min(16 * ts + (n & 7) + 8 * ab, M - 1)) * (uint32_t)K * 2u +
                             (BITS == 4 ? (uint32_t)(n >> 3) * 64u + (uint32_t)q * 16u   // step pair: first 64 bytes | second
                                        : (uint32_t)q * 32u + (uint32_t)(n >> 3) * 16u);  // group: first 16 of the lane's 32 | second

    const uint32_t mask = opaque_s(ANY ? kMask16 : kNibbleMask);
    const uint32_t magic = opaque_v(ANY ? kMagic16 : kMagic128);
    const uint32_t ones = 0x3f803f80u;
    // picks element q of four bf16 values in two registers, twice
    const uint32_t sel_q = 0x01000100u + 0x02020202u * (uint32_t)q;

    auto transpose = [](uint32_t& s0, uint32_t& s1, uint32_t& s2, uint32_t& s3) {
        const auto p = __builtin_amdgcn_permlane16_swap(s0, s1, false, false);
        const auto r = __builtin_amdgcn_permlane16_swap(s2, s3, false, false);
        const auto e = __builtin_amdgcn_permlane32_swap(p[0], r[0], false, false);
        const auto o = __builtin_amdgcn_permlane32_swap(p[1], r[1], false, false);
        s0 = e[0];
        s1 = o[0];
        s2 = e[1];
        s3 = o[1];
    };

    auto swap_halves = [](uint4& e, uint4& o) {  // the even step's upper 32 lanes against the odd step's lower ones
        const auto x = __builtin_amdgcn_permlane32_swap(e.x, o.x, false, false);
        const auto y = __builtin_amdgcn_permlane32_swap(e.y, o.y, false, false);
        const auto z = __builtin_amdgcn_permlane32_swap(e.z, o.z, false, false);
        const auto w = __builtin_amdgcn_permlane32_swap(e.w, o.w, false, false);
        e = make_uint4(x[0], y[0], z[0], w[0]);
        o = make_uint4(x[1], y[1], z[1], w[1]);
    };

    f32x4_t acc[RS][TS];
#pragma unroll
    for (int rs = 0; rs < RS; rs++)
#pragma unroll
        for (int ts = 0; ts < TS; ts++) acc[rs][ts] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};

    uint4* const sbq = reinterpret_cast<uint4*>(lds_raw);
    const int sb_pitch = quads + 1;

    // Scales and biases of the workgroup's rows: fetched once by all threads together, whole rows (every wavefront
    // fetching its own 8 bytes per row and run cost as much time as the weights), into LDS as (s0 s1, s2 s3, b0 b1,
    // b2 b3) per row and run; rows are a run apart plus 16 bytes, so that the 16 rows a wavefront reads at once fall into
    // different banks.  The loads go out first, the first pass's x and weights behind them, and only then are they stored.
    constexpr int NT = NW * kWave;
    constexpr int PRE = ANY ? 2 : tok16_stage_pieces(NW);
    [[maybe_unused]] const int pieces = ROWS * quads;
    [[maybe_unused]] uint2 sv[PRE], bv[PRE];
    // ANY: the flat scales, then the flat biases of rows row0 .. row0 + have - 1, eight values a piece
    const int sgroups = ANY ? K >> a.gs_shift : groups;
    const int have = min(OUTS, N - row0);
    const uint32_t flat = (uint32_t)have * (uint32_t)sgroups, part_pieces = (flat + 7) >> 3;
    const uint32_t all_pieces = 2u * PAIRS * part_pieces;  // (PAIR: then those of the up matrix)
    [[maybe_unused]] uint4 fv[PRE];
    auto load_flat = [&](uint32_t p) {
        uint32_t part = p >= part_pieces ? 1u : 0u;
        if (PAIR) part = p / part_pieces;
        const uint32_t e = (p - part * part_pieces) * 8u;
        const gptr_t base = (PAIR && part >= 2u ? (part & 1u ? bg2 : sg2) : (part & 1u ? bg : sg)) + (size_t)row0 * (size_t)sgroups * 2u;
        if (e + 8u <= flat) return load_u128_at(base, e * 2u);
        uint32_t v[4] = {0u, 0u, 0u, 0u};  // the last rows of the matrix end inside the piece
        for (uint32_t i = 0; e + i < flat; i++)
            v[i >> 1] |= (uint32_t)*reinterpret_cast<const __attribute__((address_space(1))) uint16_t*>(base + (e + i) * 2u) << (16u * (i & 1u));
        return make_uint4(v[0], v[1], v[2], v[3]);
    };
    auto store_flat = [&](uint32_t p, const uint4& v) {
        uint16_t* const lds16 = reinterpret_cast<uint16_t*>(lds_raw);
        uint32_t part = p >= part_pieces ? 1u : 0u;
        if (PAIR) part = p / part_pieces;
        const uint32_t e = (p - part * part_pieces) * 8u, second = part & 1u;
        uint32_t r = e / (uint32_t)sgroups, g = e - r * (uint32_t)sgroups;
        r += (part >> 1) * OUTS;
        if (G32 && (sgroups & 7) == 0) {  // whole runs: the piece is the scales (or biases) of one run of one row
            sbq[(r * (uint32_t)sb_pitch + (g >> 3)) * 2u + second] = v;
            return;
        }
        const uint32_t w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
        for (uint32_t i = 0; i < 8; i++) {
            const uint16_t h = (uint16_t)(w[i >> 1] >> (16u * (i & 1u)));
            const uint32_t run = (r * (uint32_t)sb_pitch * 2u + second) * GPR;
            if (e + i < flat) {
                if (!G32 && a.gs_shift == 7) {  // groups of 128 fill two places of 64
                    lds16[run + (g >> 1) * (2u * GPR) + 2u * (g & 1u)] = h;
                    lds16[run + (g >> 1) * (2u * GPR) + 2u * (g & 1u) + 1u] = h;
                } else {
                    lds16[run + g / GPR * (2u * GPR) + g % GPR] = h;
                }
            }
            const bool wrap = g + 1 == (uint32_t)sgroups;
            g = wrap ? 0u : g + 1;
            r += wrap ? 1u : 0u;
        }
    };
    if constexpr (ANY) {
#pragma unroll
        for (int i = 0; i < PRE; i++)
            if ((uint32_t)(tid + i * NT) < all_pieces) fv[i] = load_flat((uint32_t)(tid + i * NT));
    } else {
#pragma unroll
        for (int i = 0; i < PRE; i++) {
            const int p = tid + i * NT;
            if (p < pieces) {
                const int r = p / quads, c = p - r * quads;
                const uint32_t at = (uint32_t)min(row0 + r % OUTS, N - 1) * (uint32_t)groups * 2u + (uint32_t)c * 8u;
                sv[i] = load_u64_at(PAIR && r >= OUTS ? sg2 : sg, at);
                bv[i] = load_u64_at(PAIR && r >= OUTS ? bg2 : bg, at);
            }
        }
    }
    __builtin_amdgcn_sched_barrier(0);

    // A pass: QW runs of this wavefront (NW runs apart), their A operands in registers, and the RS sets of rows streamed
    // past them one set at a time through a ring of RING register slots.  Loads return in the order they were issued, and
    // requests that are out at the same time come back in the order the memory likes, not in the order they are needed:
    // a set is therefore requested only RING sets ahead of its use, which keeps HBM busy during the arithmetic without
    // making the first set wait for the last.
    uint4 ring[RING][QW][LINES][2];
    auto issue_set = [&](auto slot_tag, int rs_dyn, const int (&qds)[QW]) {
        constexpr int SL = decltype(slot_tag)::value;
#pragma unroll
        for (int j = 0; j < QW; j++)
#pragma unroll
            for (int ln = 0; ln < LINES; ln++)
#pragma unroll
                for (int ab = 0; ab < 2; ab++) {
                    uint32_t base = 0;
#pragma unroll
                    for (int rs = 0; rs < RS; rs++) base = rs == rs_dyn ? w_lane[rs][ab] : base;
                    const uint32_t in_row = (uint32_t)qds[j] * (uint32_t)(128 * LINES) + (uint32_t)ln * 128u;
                    ring[SL][j][ln][ab] = load_u128_stream_at(PAIR && rs_dyn >= RS / 2 ? wg2 : wg, base + (ANY ? min(in_row + w_part, row_bytes - 16u) : in_row));
                }
    };
    bool staged = false;
    // ANY: the places of LDS that no scale or bias fills (behind the end of K in a row's last run) hold zeros
    auto clear_rest = [&]() {
        uint16_t* const lds16 = reinterpret_cast<uint16_t*>(lds_raw);
        const int first = K / GRP - (quads - 1) * GPR;  // first empty place of the last run
        for (int i = tid; first < GPR && i < ROWS * 2; i += NT)
            for (int g = first; g < GPR; g++) lds16[(((i >> 1) * (quads + 1) + quads - 1) * 2 + (i & 1)) * GPR + g] = 0;
    };
    // (ANY: a wavefront without a run of its own goes through the loop once as well, to take its share of the staging)
    for (int qbase = wave; qbase < quads || (ANY && qbase == wave); qbase += NW * QW) {
        int qds[QW];   // clamped: a run past the end of K is loaded from the last run and not used
        bool live[QW];
#pragma unroll
        for (int j = 0; j < QW; j++) {
            live[j] = qbase + j * NW < quads;
            qds[j] = live[j] ? qbase + j * NW : ANY ? 0 : qbase;
        }
        uint4 xa[TS][QW][4], xb[TS][QW][4];
#pragma unroll
        for (int ts = 0; ts < TS; ts++)
#pragma unroll
            for (int j = 0; j < QW; j++)
#pragma unroll
                for (int sp = 0; sp < 4; sp++) {
                    const bool inside = !ANY || qds[j] * 256 + sp * 64 < K;  // uniform
                    const uint32_t in_row = inside ? (uint32_t)qds[j] * 512u + (uint32_t)sp * 128u : 0u;
                    xa[ts][j][sp] = load_u128_at(xg, x_lane[ts][0] + in_row);
                    xb[ts][j][sp] = load_u128_at(xg, x_lane[ts][1] + in_row);
                }
        __builtin_amdgcn_sched_barrier(0);
        issue_set(std::integral_constant<int, 0>{}, 0, qds);
        if constexpr (RING > 1 && RS > 1) issue_set(std::integral_constant<int, 1 % RING>{}, 1, qds);
        if constexpr (RING > 2 && RS > 2) issue_set(std::integral_constant<int, 2 % RING>{}, 2, qds);
        __builtin_amdgcn_sched_barrier(0);
        if (ANY && !staged) {
#pragma unroll
            for (int i = 0; i < PRE; i++)
                if ((uint32_t)(tid + i * NT) < all_pieces) store_flat((uint32_t)(tid + i * NT), fv[i]);
            for (uint32_t p = (uint32_t)(tid + PRE * NT); p < all_pieces; p += NT) store_flat(p, load_flat(p));
            clear_rest();
            __syncthreads();
            staged = true;
        }
        if (!ANY && !staged) {
#pragma unroll
            for (int i = 0; i < PRE; i++) {
                const int p = tid + i * NT;
                if (p < pieces) {
                    const int r = p / quads, c = p - r * quads;
                    sbq[r * sb_pitch + c] = make_uint4(sv[i].x, sv[i].y, bv[i].x, bv[i].y);
                }
            }
            __syncthreads();
            staged = true;
        }

        if (ANY && !live[0]) break;

        // A operands of the pass's runs, and per run the three-way split of the lane block's group sum of x
        bf16x8_t af[TS][QW][8], a2[TS][QW][GPR / 4];
#pragma unroll
        for (int ts = 0; ts < TS; ts++)
#pragma unroll
        for (int j = 0; j < QW; j++) {
            if (ANY && (qds[j] + 1) * 256 > K) {
#pragma unroll
                for (int sp = 0; sp < 4; sp++)
                    if (qds[j] * 256 + sp * 64 >= K) xa[ts][j][sp] = xb[ts][j][sp] = make_uint4(0u, 0u, 0u, 0u);
            }
            float ps[GPR];
            uint4 held = {0u, 0u, 0u, 0u};  // 8 bit, groups of 32: the even step, until the odd one is there to swap with
#pragma unroll
            for (int st = 0; st < 8; st++) {
                // even step: lanes i >= 8 take tokens 8..15 from the second load's lanes i - 8; odd step: lanes i < 8 take
                // tokens 0..7 from the first load's lanes i + 8
                const uint4 va = xa[ts][j][st >> 1], vb = xb[ts][j][st >> 1];
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
                if constexpr (BITS == 8 && G32) {
                    if ((st & 1) == 0) {
                        held = v;
                        continue;
                    }
                    swap_halves(held, v);
                    af[ts][j][st - 1] = as_bf16x8(held.x, held.y, held.z, held.w);
                    float hs = dot2_bf16(held.x, ones, 0.0f);
                    hs = dot2_bf16(held.y, ones, hs);
                    hs = dot2_bf16(held.z, ones, hs);
                    ps[st - 1] = dot2_bf16(held.w, ones, hs);
                }
                if constexpr (BITS == 4) {  // the order the expansion leaves the codes of a word in: 0 4 1 5 2 6 3 7
                    af[ts][j][st] = as_bf16x8(__builtin_amdgcn_perm(v.z, v.x, 0x05040100u), __builtin_amdgcn_perm(v.z, v.x, 0x07060302u),
                                              __builtin_amdgcn_perm(v.w, v.y, 0x05040100u), __builtin_amdgcn_perm(v.w, v.y, 0x07060302u));
                } else {
                    af[ts][j][st] = as_bf16x8(v.x, v.y, v.z, v.w);
                }
                float hs = !G32 && (st & 1) ? ps[st >> 1] : 0.0f;
                hs = dot2_bf16(v.x, ones, hs);
                hs = dot2_bf16(v.y, ones, hs);
                hs = dot2_bf16(v.z, ones, hs);
                hs = dot2_bf16(v.w, ones, hs);
                ps[G32 ? st : st >> 1] = hs;
            }
            // block q of register g holds lane block q's share of group g; transposed, the four registers of block q are
            // the four shares of group q
#pragma unroll
            for (int g4 = 0; g4 < GPR / 4; g4++) {
            uint32_t t0 = __float_as_uint(ps[4 * g4]), t1 = __float_as_uint(ps[4 * g4 + 1]), t2 = __float_as_uint(ps[4 * g4 + 2]),
                     t3 = __float_as_uint(ps[4 * g4 + 3]);
            transpose(t0, t1, t2, t3);
            float X = (__uint_as_float(t0) + __uint_as_float(t1)) + (__uint_as_float(t2) + __uint_as_float(t3));
            if (!live[j]) X = 0.0f;
            X *= kUnit;
            const uint32_t u0 = __float_as_uint(X) & 0xffff0000u;
            const float r1 = X - __uint_as_float(u0);
            const uint32_t u1 = __float_as_uint(r1) & 0xffff0000u;
            const float r2 = r1 - __uint_as_float(u1);
            const uint32_t u2 = __float_as_uint(r2) & 0xffff0000u;
            const uint32_t m0 = __float_as_uint(kLacks * __uint_as_float(u0));
            const uint32_t m1 = __float_as_uint(kLacks * __uint_as_float(u1));
            const uint32_t m2 = __float_as_uint(kLacks * __uint_as_float(u2));
            a2[ts][j][g4] = as_bf16x8((u0 >> 16) | u1, (u2 >> 16) | m0, (m1 >> 16) | m2, 0u);
            }
        }

        auto run_set = [&](auto rs_tag) {
            constexpr int rs = decltype(rs_tag)::value;
            constexpr int SL = rs % RING;
#pragma unroll
            for (int j = 0; j < QW; j++) {
                // first 64 bytes of all 16 rows (lanes i >= 8 from the second load's lanes i - 8), second 64 bytes (lanes
                // i < 8 from the first load's lanes i + 8): as for x
                uint32_t ww[8 * LINES];  // 4 bit: the word of step st; 8 bit: the two words of step st at 2 st, 2 st + 1
#pragma unroll
                for (int ln = 0; ln < LINES; ln++) {
                    const uint4 la = ring[SL][j][ln][0], lb = ring[SL][j][ln][1];
                    uint32_t f0 = __builtin_amdgcn_update_dpp(la.x, lb.x, 0x118, 0xf, 0xc, false);
                    uint32_t f1 = __builtin_amdgcn_update_dpp(la.y, lb.y, 0x118, 0xf, 0xc, false);
                    uint32_t f2 = __builtin_amdgcn_update_dpp(la.z, lb.z, 0x118, 0xf, 0xc, false);
                    uint32_t f3 = __builtin_amdgcn_update_dpp(la.w, lb.w, 0x118, 0xf, 0xc, false);
                    uint32_t g0 = __builtin_amdgcn_update_dpp(lb.x, la.x, 0x108, 0xf, 0x3, false);
                    uint32_t g1 = __builtin_amdgcn_update_dpp(lb.y, la.y, 0x108, 0xf, 0x3, false);
                    uint32_t g2 = __builtin_amdgcn_update_dpp(lb.z, la.z, 0x108, 0xf, 0x3, false);
                    uint32_t g3 = __builtin_amdgcn_update_dpp(lb.w, la.w, 0x108, 0xf, 0x3, false);
                    if constexpr (BITS == 4) {
                        transpose(f0, f1, f2, f3);
                        transpose(g0, g1, g2, g3);
                    }
                    const uint32_t both[8] = {f0, f1, f2, f3, g0, g1, g2, g3};
#pragma unroll
                    for (int k = 0; k < 8; k++) ww[8 * ln + k] = both[k];
                }
                if constexpr (BITS == 8 && G32) {
#pragma unroll
                    for (int g = 0; g < 4; g++)
#pragma unroll
                        for (int k = 0; k < 2; k++) {
                            const auto p = __builtin_amdgcn_permlane32_swap(ww[4 * g + k], ww[4 * g + 2 + k], false, false);
                            ww[4 * g + k] = p[0];
                            ww[4 * g + 2 + k] = p[1];
                        }
                }
                // scales, then biases, of the run's groups (groups of 32: 16 bytes each)
                uint4 sbv, bbv;
                if constexpr (G32) {
                    sbv = sbq[((rs * 16 + n) * sb_pitch + qds[j]) * 2];
                    bbv = sbq[((rs * 16 + n) * sb_pitch + qds[j]) * 2 + 1];
                } else {
                    sbv = sbq[(rs * 16 + n) * sb_pitch + qds[j]];
                    bbv = make_uint4(sbv.z, sbv.w, 0u, 0u);
                }
                f32x4_t part[TS];
#pragma unroll
                for (int ts = 0; ts < TS; ts++) part[ts] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
                for (int g = 0; g < 4; g++) {
                    f32x4_t d[TS];
#pragma unroll
                    for (int ts = 0; ts < TS; ts++) d[ts] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
                    for (int half = 0; half < 2; half++) {
                        uint32_t e[4];
                        if constexpr (BITS == 4 && CENTRED) {
                            unpack4_centred(ww[2 * g + half], e);
                        } else if constexpr (BITS == 4 && ANY) {
                            const uint4 v = unpack_word4(ww[2 * g + half], mask, magic);
                            e[0] = v.x, e[1] = v.y, e[2] = v.z, e[3] = v.w;
                        } else if constexpr (BITS == 4) {
                            unpack4_word(ww[2 * g + half], mask, magic, e);
                        } else if constexpr (CENTRED) {
                            unpack8_centred(ww[4 * g + 2 * half], e);
                            unpack8_centred(ww[4 * g + 2 * half + 1], e + 2);
                        } else {
                            unpack8_word(ww[4 * g + 2 * half], e);
                            unpack8_word(ww[4 * g + 2 * half + 1], e + 2);
                        }
                        const bf16x8_t bop = as_bf16x8(e[0], e[1], e[2], e[3]);
                        if constexpr (G32) {  // a step is a group
                            const uint32_t sw = g == 0 ? sbv.x : g == 1 ? sbv.y : g == 2 ? sbv.z : sbv.w;
                            const float sc = half ? __uint_as_float(sw & 0xffff0000u) : __uint_as_float(sw << 16);
                            const f32x4_t zero = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
                            for (int ts = 0; ts < TS; ts++) {
                                const f32x4_t dg = __builtin_amdgcn_mfma_f32_16x16x32_bf16(af[ts][j][2 * g + half], bop, zero, 0, 0, 0);
#pragma unroll
                                for (int r = 0; r < 4; r++) part[ts][r] = __builtin_fmaf(sc, dg[r], part[ts][r]);
                            }
                        } else {
#pragma unroll
                            for (int ts = 0; ts < TS; ts++)
                                d[ts] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(af[ts][j][2 * g + half], bop, d[ts], 0, 0, 0);
                        }
                    }
                    if constexpr (G32) continue;
                    const uint32_t sw = g < 2 ? sbv.x : sbv.y;
                    const float sc = (g & 1) ? __uint_as_float(sw & 0xffff0000u) : __uint_as_float(sw << 16);
#pragma unroll
                    for (int ts = 0; ts < TS; ts++)
#pragma unroll
                        for (int r = 0; r < 4; r++) part[ts][r] = __builtin_fmaf(sc, d[ts][r], part[ts][r]);
                }
#pragma unroll
                for (int g4 = 0; g4 < GPR / 4; g4++) {
                    const uint32_t bb = __builtin_amdgcn_perm(g4 ? bbv.w : bbv.y, g4 ? bbv.z : bbv.x, sel_q);
                    const uint32_t ss = __builtin_amdgcn_perm(g4 ? sbv.w : sbv.y, g4 ? sbv.z : sbv.x, sel_q);
                    const bf16x8_t b2 = as_bf16x8(bb, __builtin_amdgcn_perm(ss, bb, 0x05040100u), ss, 0u);
#pragma unroll
                    for (int ts = 0; ts < TS; ts++)
                        part[ts] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a2[ts][j][g4], b2, part[ts], 0, 0, 0);
                }
                // a run past the end of K (x and weights of the last run were loaded in its place) adds nothing
                if (live[j]) {
#pragma unroll
                    for (int ts = 0; ts < TS; ts++)
#pragma unroll
                        for (int r = 0; r < 4; r++) acc[rs][ts][r] += part[ts][r];
                }
            }
            if constexpr (rs + RING < RS) {
                __builtin_amdgcn_sched_barrier(0);
                issue_set(std::integral_constant<int, SL>{}, rs + RING, qds);
                __builtin_amdgcn_sched_barrier(0);
            }
        };
        run_set(std::integral_constant<int, 0>{});
        if constexpr (RS > 1) run_set(std::integral_constant<int, 1>{});
        if constexpr (RS > 2) run_set(std::integral_constant<int, 2>{});
        if constexpr (RS > 3) run_set(std::integral_constant<int, 3>{});
        static_assert(RS <= 4, "sets of rows per workgroup");
    }
    if (!ANY && !staged) __syncthreads();  // a wavefront without a run of its own

    // ---- the wavefronts' partial sums meet in LDS: red[wave][token][row]; thread (token, row) adds them in wave order ----
    // (behind the staged scales and biases: a wavefront may get here while another still reads those)
    float* red = reinterpret_cast<float*>(lds_raw + (ANY ? 0 : (size_t)ROWS * sb_pitch * 16));
    if constexpr (ANY) __syncthreads();  // (the scales of long rows in groups of 32 leave no room: in their place)
    // D layout of the 16x16 MFMA: lane (n, q), register r -> token 4 q + r (of its set), weight row n
#pragma unroll
    for (int rs = 0; rs < RS; rs++)
#pragma unroll
        for (int ts = 0; ts < TS; ts++)
#pragma unroll
            for (int r = 0; r < 4; r++) red[(wave * 16 * TS + 16 * ts + 4 * q + r) * TSTRIDE + rs * 16 + n] = acc[rs][ts][r];
    __syncthreads();
    auto total_of = [&](int t, int column) {
        float total = red[t * TSTRIDE + column];
#pragma unroll
        for (int p = 1; p < NW; p++) total += red[(p * 16 * TS + t) * TSTRIDE + column];
        return kUnit != 1.0f ? total * (1.0f / kUnit) : total;
    };
    for (int o = tid; o < 16 * TS * OUTS; o += NW * kWave) {
        const int t = o / OUTS, rl = o - t * OUTS;
        const int row = row0 + rl;
        if (t >= M || row >= N) continue;
        float total = total_of(t, rl);
        [[maybe_unused]] float up = PAIR ? total_of(t, OUTS + rl) : 0.0f;
        if constexpr (G32 && !GROUPED) {  // (dense groups of 32 keep what the any-width kernel makes of infinities)
#pragma nounroll
            for (int part = 0; part < PAIRS; part++) {
                if (!not_finite(part ? up : total)) continue;
                const float v = plain_dot_g32(a.x + (size_t)t * K, (PAIR && part ? a.w2 : a.w) + (size_t)row * (row_bytes / 4),
                                              (PAIR && part ? a.s2 : a.s) + (size_t)row * sgroups, (PAIR && part ? a.b2 : a.b) + (size_t)row * sgroups, K, BITS);
                if (part) up = v; else total = v;
            }
        }
        if constexpr (PAIR) total = fmul_unfused(act_value(a.act, total), up);
        size_t y_row = (size_t)t;
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
}

template <int BITS, int RS, int RING, int TS, bool ANY, int GRP, bool PAIR>
__global__ __launch_bounds__(kTokWaves* kWave) void qmv_tok16_kernel(const QmvArgs a) {
    qmv_tok16_body<BITS, kTokWaves, RS, 1, RING, TS, ANY, GRP, PAIR, false>(a, (int)blockIdx.x);
}
template <int BITS, int RS, int RING, int TS, int GRP, bool PAIR>
__global__ __launch_bounds__(kTokWaves* kWave) void qmv_tok16_grouped_kernel(const QmvArgs a) {
    qmv_tok16_body<BITS, kTokWaves, RS, 1, RING, TS, true, GRP, PAIR, true>(a, (int)blockIdx.x);
}
// up to four matrices that share x in one grid: every workgroup belongs to one of them
template <int BITS, int RS, int RING, int TS, bool ANY, int GRP>
__global__ __launch_bounds__(kTokWaves* kWave) void qmv_tok16_multi_kernel(const QmvMultiArgs ma) {
    int i = 0, before = 0;
    while (i + 1 < ma.count && (int)blockIdx.x >= ma.block_end[i]) before = ma.block_end[i++];
    QmvArgs a = ma.common;
    a.w = ma.w[i];
    a.s = ma.s[i];
    a.b = ma.b[i];
    a.y = ma.y[i];
    a.N = ma.N[i];
    qmv_tok16_body<BITS, kTokWaves, RS, 1, RING, TS, ANY, GRP, false, false>(a, (int)blockIdx.x - before);
}

// ---- kernels of one code width -------------------------------------------------------------------------------------

typedef void (*QmvTokKernel)(const QmvArgs);
typedef void (*QmvTokMultiKernel)(const QmvMultiArgs);
// forms of the kernel: groups of 64 with K a multiple of 256; groups of 64 or 128 with K a multiple of 64; groups of 32
enum { kTokExact = 0, kTokAny = 1, kTokG32 = 2, kTokForms = 3 };
struct QmvTokEntry {
    QmvVariant v;  // m = most activation rows, rows = sets of weight rows per workgroup, waves = wavefronts that share K
                   // (depth = sets of rows in flight, xmode = runs of 256 codes a wavefront holds per pass)
    QmvTokKernel fn[kTokForms];
    QmvTokMultiKernel multi[kTokForms];
    QmvTokKernel pair[kTokForms];     // null for one set of rows per workgroup
    QmvTokKernel grouped[2][2];       // [groups of 32][pair], four sets of rows only
    const char* name[kTokForms];
    int wg_rows;  // weight rows per workgroup
    int lds;      // bytes of the partial sums
};
// TS: sets of 16 tokens per expanded weight (1: up to 16 rows of x, 2: up to 32)
#define AQ_QMVT_(BITS, TAG, M, RS, RING, TS, PAIRS, GROUPED)                                                             \
    {                                                                                                                    \
        {"qmvt_b" #BITS "_m" TAG "_r" #RS "_w8_q1_d" #RING, BITS, M, RS, 8, RING, 0, 1, 6},                               \
            {qmv_tok16_kernel<BITS, RS, RING, TS, false, 64, false>, qmv_tok16_kernel<BITS, RS, RING, TS, true, 64, false>, \
             qmv_tok16_kernel<BITS, RS, RING, TS, true, 32, false>},                                                      \
            {qmv_tok16_multi_kernel<BITS, RS, RING, TS, false, 64>, qmv_tok16_multi_kernel<BITS, RS, RING, TS, true, 64>,  \
             qmv_tok16_multi_kernel<BITS, RS, RING, TS, true, 32>},                                                       \
            PAIRS(BITS, RS, RING, TS), GROUPED(BITS, RS, RING, TS),                                                       \
            {"qmvt_b" #BITS "_m" TAG "_r" #RS "_w8_q1_d" #RING, "qmvt_b" #BITS "_m" TAG "_r" #RS "_any",                   \
             "qmvt_b" #BITS "_m" TAG "_r" #RS "_s32"},                                                                    \
            16 * RS, 8 * 16 * TS * (16 * RS) * 4                                                                          \
    }
#define AQ_QMVT_NOPAIR(BITS, RS, RING, TS) {nullptr, nullptr, nullptr}
#define AQ_QMVT_PAIR(BITS, RS, RING, TS)                                                                     \
    {                                                                                                        \
        qmv_tok16_kernel<BITS, RS, RING, TS, false, 64, true>, qmv_tok16_kernel<BITS, RS, RING, TS, true, 64, true>, \
            qmv_tok16_kernel<BITS, RS, RING, TS, true, 32, true>                                              \
    }
#define AQ_QMVT_NOGROUP(BITS, RS, RING, TS) {{nullptr, nullptr}, {nullptr, nullptr}}
#define AQ_QMVT_GROUP(BITS, RS, RING, TS)                                                                    \
    {                                                                                                        \
        {qmv_tok16_grouped_kernel<BITS, RS, RING, TS, 64, false>, qmv_tok16_grouped_kernel<BITS, RS, RING, TS, 64, true>}, \
        {                                                                                                    \
            qmv_tok16_grouped_kernel<BITS, RS, RING, TS, 32, false>, qmv_tok16_grouped_kernel<BITS, RS, RING, TS, 32, true> \
        }                                                                                                    \
    }
#define AQ_QMVT_SET(BITS)                                                                                    \
    AQ_QMVT_(BITS, "16", 16, 4, 2, 1, AQ_QMVT_PAIR, AQ_QMVT_GROUP), AQ_QMVT_(BITS, "16", 16, 2, 2, 1, AQ_QMVT_PAIR, AQ_QMVT_NOGROUP), \
        AQ_QMVT_(BITS, "16", 16, 1, 1, 1, AQ_QMVT_NOPAIR, AQ_QMVT_NOGROUP),                                    \
        AQ_QMVT_(BITS, "32_s2", 32, 4, 2, 2, AQ_QMVT_PAIR, AQ_QMVT_GROUP),                                     \
        AQ_QMVT_(BITS, "32_s2", 32, 2, 2, 2, AQ_QMVT_PAIR, AQ_QMVT_NOGROUP),                                   \
        AQ_QMVT_(BITS, "32_s2", 32, 1, 1, 2, AQ_QMVT_NOPAIR, AQ_QMVT_NOGROUP)

constexpr int kTokPerWidth = 6;
const QmvTokEntry* tok_entries_4();  // aq_qmv_tok.hip
const QmvTokEntry* tok_entries_8();  // aq_qmv_tok8.hip (a source of its own: compile time)

}  // namespace aq
