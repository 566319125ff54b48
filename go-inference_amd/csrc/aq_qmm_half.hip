// affine_qmm for gfx950, prefill sizes, fp16 matrix-core operands; 4-bit codes: the scale rides inside the operand (8-bit
// codes: see BITS 8 at the kernel).
//
// Same contract as the tile kernels of aq_qmm_tile.hip (MLX affine_qmm_t,
// go/engine/metal/quant_seam_backend.go:77-109; replaces rocm_mlx_q4_projection_batch*,
// go/engine/hip/kernels/quant/affine_projection_tuned.hipinc:166-1109).  Those multiply x with the bare codes
// and pay one fp32 FMA per output element and 64-code block to apply the scale, which keeps the accumulators
// in vector registers and the vector unit as busy as the matrix cores.  Here
//
//     w = scale * code + bias = scale * (code - 8) + (bias + 8 * scale)
//
// and scale * (code - 8) is formed EXACTLY as an fp16 value: a bf16 scale has 8 significant bits, |code - 8| <= 8
// has at most 3 below its leading one, so the product has at most 11 - what fp16 holds.  It is produced by one
// packed fp16 FMA per two codes, (16 + code) * s - 24 * s, with 16 + code built by OR-ing the nibble into the
// mantissa of fp16 16.0 and 24 * s exact (24 = 3 * 8).  The activations are bf16 and therefore exact in fp16 too,
// given the exponent range, which two power-of-two factors take care of: every row of x is scaled so that its
// largest magnitude lies in [2^14, 2^15) and every row of the weights so that its largest scale lies in
// [2^10, 2^11) (elements more than 2^28 below their row's largest lose low bits to fp16's subnormal range: far
// below the fp32 accumulation noise).  The matrix cores then accumulate x * w over all of K with no vector work
// on the accumulators at all, the epilogue multiplies by the two inverse powers of two, and the affine term
// (bias + 8 * scale) * sum(x) still costs one bf16 MFMA per four blocks as in the tile kernels.
// What is left for the vector unit is the expansion of the codes: 12 instructions per packed word, amortised
// over 128 rows of x per wavefront (wavefront tiles 128 x 64: 32 MFMAs per 64-code block, about three vector
// instructions each).
//
// Operand staging is that of the tile kernels: activations rewritten once in A-fragment order (here as fp16,
// one workgroup per row so that the row's largest magnitude is known), A tiles and PACKED weights copied
// global -> LDS by copy instructions three blocks deep, one barrier per block, XCD-aware tile order.
#include "aq_device.h"
#include "aq_fp16_operands.h"
#include "aq_kernels.h"
#include "aq_lds_copy.h"
#include "aq_qmm.h"
#include "aq_share_sum.h"

#include <algorithm>
#include <cmath>
#include <type_traits>

namespace aq {

namespace {

typedef _Float16 f16x2_t __attribute__((ext_vector_type(2)));
typedef _Float16 f16x8_t __attribute__((ext_vector_type(8)));

constexpr uint32_t kMaskH = 0x03C003C0u;   // a nibble moved to fp16 mantissa bits [9:6]
constexpr uint32_t kMagicH = 0x4C004C00u;  // fp16 16.0 in both halves: 16 + code, exact

// Pair I (codes I and I + 4) of a packed word -> fp16 values s * (code - 8); the pairs of a word in order are its slot order
// (c0,c4)(c1,c5)(c2,c6)(c3,c7)
template <int I>
__device__ __forceinline__ uint32_t expand_pair(uint32_t w, uint32_t mask_s, uint32_t magic_v, f16x2_t s2, f16x2_t m24) {
    const uint32_t at = I == 0 ? w << 6 : I == 1 ? w << 2 : I == 2 ? w >> 2 : w >> 6;
    return __builtin_bit_cast(uint32_t, __builtin_elementwise_fma(__builtin_bit_cast(f16x2_t, and_or(at, mask_s, magic_v)), s2, m24));
}

// 8 codes of two packed words of 8-bit codes -> 8 fp16 values code - 128 in their natural order: the bytes go into the
// mantissa of fp16 1024.0, whose unit in the last place is 1, and 1152 comes off again; both steps are exact
__device__ __forceinline__ f16x8_t expand_bytes(uint2 w) {
    const f16x2_t off = {(_Float16)-1152.0f, (_Float16)-1152.0f};
    auto two = [&](uint32_t v, uint32_t sel) {
        return __builtin_bit_cast(uint32_t, __builtin_bit_cast(f16x2_t, __builtin_amdgcn_perm(0x64646464u, v, sel)) + off);
    };
    const uint4 u = {two(w.x, 0x04010400u), two(w.x, 0x04030402u), two(w.y, 0x04010400u), two(w.y, 0x04030402u)};
    return __builtin_bit_cast(f16x8_t, u);
}

typedef uint16_t u16x2_t __attribute__((ext_vector_type(2)));
__device__ __forceinline__ uint32_t max_u16x2(uint32_t a, uint32_t b) {
    return __builtin_bit_cast(uint32_t, __builtin_elementwise_max(__builtin_bit_cast(u16x2_t, a), __builtin_bit_cast(u16x2_t, b)));
}

// Elements off .. off + 7 of an array of `total`; what lies past its end is anything.  Rows of scales start at any even address
// (K of 704: 22 bytes a row), and one 16-byte load from there beats eight of two bytes, each of which touches as many lines.
// load_eight reads eight elements that lie inside the array, moved_down brings the asked for to the front.  (TINY: an array of
// fewer than eight.)
typedef uint32_t u32x4_at2_t __attribute__((ext_vector_type(4), aligned(2)));
template <bool TINY>
__device__ __forceinline__ uint4 load_eight(const uint16_t* base, uint32_t off, uint32_t total) {
    if constexpr (TINY) {
        uint64_t lo = 0, hi = 0;
#pragma nounroll
        for (uint32_t i = 0; i < 4; i++) {
            lo |= (uint64_t)base[min(off + i, total - 1)] << (16 * i);
            hi |= (uint64_t)base[min(off + 4 + i, total - 1)] << (16 * i);
        }
        return make_uint4((uint32_t)lo, (uint32_t)(lo >> 32), (uint32_t)hi, (uint32_t)(hi >> 32));
    }
    const u32x4_at2_t v = *reinterpret_cast<const u32x4_at2_t*>(base + min(off, total - 8));
    return make_uint4(v[0], v[1], v[2], v[3]);
}
__device__ __forceinline__ uint4 moved_down(uint4 v, uint32_t off, uint32_t total) {
    const uint32_t by = total >= 8 && off > total - 8 ? min(off - (total - 8), 7u) : 0u;
    v.x = by & 4 ? v.z : v.x;
    v.y = by & 4 ? v.w : v.y;
    v.x = by & 2 ? v.y : v.x;
    v.y = by & 2 ? v.z : v.y;
    v.z = by & 2 ? v.w : v.z;
    const uint32_t half = (by & 1) * 16;
    return make_uint4(__builtin_amdgcn_alignbit(v.y, v.x, half), __builtin_amdgcn_alignbit(v.z, v.y, half), __builtin_amdgcn_alignbit(v.w, v.z, half),
                      v.w >> half);
}

}  // namespace

// ---- pass over x ----------------------------------------------------------------------------
// One workgroup per ROWS rows of x (rows padded to a multiple of 32 are written as zeros).  Thread (r = tid % ROWS, p = tid /
// ROWS) works on 16-byte pieces p, p + 512 / ROWS, ... of row r.  The slots of eight rows in a fragment are one 128-byte line;
// with fewer rows a workgroup the others' run on the same XCD at about the same time, so that a line is put together in its L2
// (spread over the XCDs two rows a workgroup took 33 us for 2048 x 15360, one row 56; here 22 and 32).
// Bound: latency of two dependent passes in few workgroups, then memory (2048 x 15360: 126 MB in 22 us, 5.7 TB/s).  Eight rows a
// workgroup from 1024 rows on, one below, magnitudes and block sums value by value -> here (us): 509 x 3840 8.0 -> 6.1, 509 x
// 15360 16.8 -> 10.2, 777 x 10240 17.6 -> 10.1, 1024 x 15360 35.8 -> 13.3, 2048 x 4096 11.9 -> 9.9, 2048 x 15360 37.8 -> 22.4.
// xf: [mblks][K/16][64 lanes][8] fp16, the A-fragment order of the tile kernels (4-bit slot order), values
//     x * 2^e with e chosen per row;
// xs: [mblks][ceil(G/4)][32 rows][4 blocks][hi, lo] bf16: 2^e * sum of x over each 64-code block, hi + lo (a wavefront's
//     load of 32 rows is four lines; row-major it was 32);
// rs: [mblks * 32] fp32: 2^-e.
//
// GRP 32: xs holds the sums of the 32-code halves, [mblks][ceil(G/4)][half][32 rows][4 blocks][hi, lo].
// GROUPED: row i of the fragments is row route_x[i] of x (the list of routes sorted by expert; negative: zeros), and rows
// past *live_rows are left alone.
// tickets: `count` words that the tiles of shared K start from at zero.
constexpr int kPrepThreads = 512;
constexpr int kPrepHold = 8;
// BITS 8: the order in which the 8-bit kernels take x: lane half h has codes 32 i + 16 h .. + 15 of a block in steps 2 i and 2 i + 1
// (one 16-byte read of the weights), values in their natural order.
template <int ROWS, int GRP, int BITS>
__global__ __launch_bounds__(kPrepThreads) void qmmh_prep_kernel(const uint16_t* __restrict__ x, uint16_t* __restrict__ xf,
                                                         uint16_t* __restrict__ xs, float* __restrict__ rs, int M, int K,
                                                         const int32_t* __restrict__ route_x, const int32_t* __restrict__ live_rows,
                                                         uint32_t* __restrict__ tickets, int count) {
    for (int i = (int)(blockIdx.x * kPrepThreads + threadIdx.x); i < count; i += (int)gridDim.x * kPrepThreads) tickets[i] = 0u;
    constexpr int STEP = kPrepThreads / ROWS;  // pieces of a row between a thread's pieces
    // the workgroups of eight rows, which fill the same lines of xf, on one XCD
    const int seq = (int)blockIdx.x >> 3, row0 = (seq / (8 / ROWS) * 8 + ((int)blockIdx.x & 7)) * 8 + seq % (8 / ROWS) * ROWS;
    if (row0 >= (M + 31) / 32 * 32 || (live_rows && row0 >= *live_rows)) return;
    const int tid = threadIdx.x;
    const int r = tid % ROWS, p0 = tid / ROWS;
    const int row = row0 + r;
    const int G = K / 64;
    const int G4 = (G + 3) / 4;
    const int pieces = K / 8;
    const int from = route_x ? (row < M ? route_x[row] : -1) : row;
    const bool live = row < M && from >= 0;
    const uint16_t* const xrow = x + (int64_t)(live ? from : 0) * K;
    __shared__ uint32_t wave_mag[kPrepThreads / kWave][ROWS];
    // kPrepHold pieces per thread are requested together; they stay in registers for the second pass if they are all there is
    uint4 hold[kPrepHold];
    auto fetch = [&](int p) {
#pragma unroll
        for (int i = 0; i < kPrepHold; i++) {
            hold[i] = make_uint4(0u, 0u, 0u, 0u);
            if (live && p + p0 + STEP * i < pieces) hold[i] = *reinterpret_cast<const uint4*>(xrow + (p + p0 + STEP * i) * 8);
        }
    };
    // the largest magnitude, two values an instruction; inf and NaN do not set the scale, so a thread that has met one goes over
    // its pieces again, value by value
    uint32_t most = 0;
    for (int p = 0; p < pieces; p += STEP * kPrepHold) {
        fetch(p);
#pragma unroll
        for (int i = 0; i < kPrepHold; i++) {
            const uint32_t w[4] = {hold[i].x, hold[i].y, hold[i].z, hold[i].w};
#pragma unroll
            for (int c = 0; c < 4; c++) most = max_u16x2(most, w[c] & 0x7fff7fffu);
        }
    }
    uint32_t mag = max(most & 0xffffu, most >> 16);
    if (mag >= 0x7f80u) {
        mag = 0;
#pragma nounroll
        for (int p = p0; p < pieces; p += STEP) {
#pragma nounroll
            for (int c = 0; c < 8; c++) {
                const uint32_t v = xrow[p * 8 + c] & 0x7fffu;
                if (v < 0x7f80u) mag = max(mag, v);
            }
        }
    }
    // the threads of a wavefront that share a row are ROWS lanes apart
    mag = max_lanes<ROWS>(mag);
    if ((tid & (kWave - 1)) < ROWS) wave_mag[tid >> 6][r] = mag;
    __syncthreads();
    mag = 0;
#pragma unroll
    for (int w = 0; w < kPrepThreads / kWave; w++) mag = max(mag, wave_mag[w][r]);
    const int e = exponent_shift(mag, 14);
    const float up = pow2f(e);
    if (tid < ROWS) rs[row] = live ? pow2f(-e) : 0.0f;

    auto emit = [&](int p, const uint4& v) {
        const int g = p >> 3, c8 = p & 7;
        float sx = 0.0f;
        sx = dot2_bf16(v.x, 0x3F803F80u, sx);
        sx = dot2_bf16(v.y, 0x3F803F80u, sx);
        sx = dot2_bf16(v.z, 0x3F803F80u, sx);
        sx = dot2_bf16(v.w, 0x3F803F80u, sx);
        // the 8 pieces of a block of this row sit in the 8 lanes ROWS apart
        sx += lane_xor<ROWS>(sx);
        sx += lane_xor<2 * ROWS>(sx);
        if (GRP == 64) sx += lane_xor<4 * ROWS>(sx);
        if ((c8 & (GRP / 8 - 1)) == 0) {
            const float scaled = sx * up;
            const uint32_t hi = f32_to_bf16_bits(scaled);
            const uint32_t lo = f32_to_bf16_bits(scaled - bf16_bits_to_f32(hi));
            const int64_t quad = (int64_t)(row >> 5) * G4 + (g >> 2);
            uint32_t* dst = reinterpret_cast<uint32_t*>(xs) + ((GRP == 64 ? quad : 2 * quad + (c8 >> 2)) * 32 + (row & 31)) * 4;
            dst[g & 3] = hi | (lo << 16);
            if (g == G - 1)
                for (int q = (g & 3) + 1; q < 4; q++) dst[q] = 0u;
        }
        const uint32_t w[4] = {v.x, v.y, v.z, v.w};
        _Float16 hv[8];
#pragma unroll
        for (int i = 0; i < 4; i++) {
            hv[2 * i] = (_Float16)(bf16_bits_to_f32(w[i] & 0xffffu) * up);
            hv[2 * i + 1] = (_Float16)(bf16_bits_to_f32(w[i] >> 16) * up);
        }
        // slot order (x0,x4)(x1,x5)(x2,x6)(x3,x7): the order in which expand_pair emits the codes of a word
        const f16x8_t o = BITS == 4 ? f16x8_t{hv[0], hv[4], hv[1], hv[5], hv[2], hv[6], hv[3], hv[7]}
                                    : f16x8_t{hv[0], hv[1], hv[2], hv[3], hv[4], hv[5], hv[6], hv[7]};
        const int t = BITS == 4 ? c8 & 3 : (c8 >> 2) * 2 + (c8 & 1), h = BITS == 4 ? c8 >> 2 : c8 >> 1 & 1;
        const int64_t frag = (int64_t)(row >> 5) * (K / 16) + g * 4 + t;
        *reinterpret_cast<f16x8_t*>(xf + (frag * 64 + h * 32 + (row & 31)) * 8) = o;
    };
    const bool held = pieces <= STEP * kPrepHold;
    for (int p = 0; p < pieces; p += STEP * kPrepHold) {
        if (!held) fetch(p);
#pragma unroll
        for (int i = 0; i < kPrepHold; i++)
            if (p + p0 + STEP * i < pieces) emit(p + p0 + STEP * i, hold[i]);
    }
}

// Output (m, n) of a matrix (pair: of the gated pair) formed again from x itself, if what is stored there is not finite: dense
// calls in groups of 32 ran on the any-width kernel, which keeps infinities (plain_dot_g32).  The test costs a prompt of 509
// tokens 4 of 420 us (3840 / 15360); rows with an infinity cost what the any-width kernel took for them.
__device__ __forceinline__ void fix_output(const QmmHalfArgs& a, const QmmSegment& seg, int m, int n) {
    const int64_t at = (int64_t)m * seg.N + n;
    if (!not_finite(a.out_f32 ? static_cast<const float*>(seg.y)[at] : bf16_bits_to_f32(static_cast<const uint16_t*>(seg.y)[at]))) return;
    const uint16_t* const x = a.x + (int64_t)m * a.K;
    const int64_t word = (int64_t)n * (a.K / 32 * a.bits), group = (int64_t)n * (a.K / 32);
    float v[2];
#pragma nounroll
    for (int i = 0; i < (a.pair ? 2 : 1); i++) {
        const QmmSegment& from = i ? a.seg[1] : seg;
        const float d = plain_dot_g32(x, from.w + word, from.s + group, from.b + group, a.K, a.bits);
        if (i) v[1] = d; else v[0] = d;
    }
    const float y = a.pair ? fmul_unfused(act_value(a.act, v[0]), v[1]) : v[0];
    if (a.out_f32)
        static_cast<float*>(seg.y)[at] = y;
    else
        static_cast<uint16_t*>(seg.y)[at] = f32_to_bf16_bits(y);
}

// Whether a tile has LDS for its rows' factors (two of the 8-bit kernels fill half a CU's with their stages).
__host__ __device__ constexpr bool half_rows_in_lds(int bits, int mb, int waves) { return !(bits == 8 && mb == 2 && waves == 4); }

// ---- main kernel ----------------------------------------------------------------------------
// SE: elements of a row of scales (and of biases) in LDS at a time.
// GRP 32: the codes a lane half h expands are those of one group (block g's half h), so that only its scale and bias differ:
// the lane half keeps its own four scales per quad; the affine term takes its own sums on the A side and two MFMAs per quad
// (sum x bias, sum x 8 scale) instead of one.
// Several matrices (a.nseg > 1): the column tiles of all of them make one grid.
// PAIR (a.pair): column block 0 of a wavefront's tile holds gate rows, column block 1 the up rows of the same outputs; the
// store is act(gate) * up, from the accumulators as they lie.
// Expert slabs (a.chunks): a row band is a chunk of up to BM places of the list of routes sorted by expert
// (aq_moe_group.hip), its weights those of the chunk's expert, its outputs the rows of y that its routes name.
// Packed weights are staged two 64-code blocks at a time.  The L1 charges a copy instruction per line it touches, about four
// clocks each: 32 bytes of each of 32 rows per instruction (one block at a time) cost 32 lines for 1 KiB, which was most of
// what the small tiles' loop took (32 x 256 tiles: 288 lines x 4 clocks of 1320 per block) and half the copies' time in the
// large ones; two blocks are 64-byte halves of sixteen rows (2048 x 4096 x 14336: 281 -> 265 us; 4096 x 4096 x 16384: 571 ->
// 558; 512 x 4096 x 16384 on 32 x 256 tiles: 155 -> 138; whole lines, four blocks at a time, measured the same on the small
// tiles and 623 us on the large ones, whose LDS addresses then are no constants).  The 16-byte pieces of a row are rotated
// against those of its neighbours (the piece a lane fetches, not the place it lands in), so that a wavefront's reads of one
// block hit all banks.
//
// BITS 8: scale * (code - 128) has 16 significant bits, more than fp16 holds, so the operand is code - 128 alone (exact) and a
// group's partial sums P are multiplied by the fp32 scale: out += scale * P, one FMA per output element and group, as in the
// tile kernels of aq_qmm_tile.hip.  Against those: two vector instructions per pair of codes instead of three, several
// matrices in one grid, the gated pair, groups of 32 and expert slabs.  A step of the MFMA is 16 consecutive codes, so that
// groups of 32 are two steps each; bytes are staged one 64-code block at a time, in as many stages as A.
// Measured (us; bf16-code tiles -> here): 2048 x 4096 x 14336 395 -> 329, a layer of 777 rows (2560 / 10240) 453 -> 332, of 400
// rows (1472 / 4032) 274 -> 125, of 300 rows in groups of 32 (2048 / 8192) 24.7 ms on the any-width kernel -> 159, 512 tokens
// through 128 experts (2816 / 704) 3692 -> 285.  Bound: with 64 rows a wavefront, 16 MFMAs a block stand against 64 vector
// instructions of expansion and 64 of scaling; with two 128 x 128 tiles on a CU a block takes 0.65 us of it for 0.23 us of matrix pipe.
// Scales and biases go through LDS as well, SE of each row at a time (a segment).  Loaded by the lanes that use them, four blocks at
// a time, every load touched a line per row, in either wavefront row again: as many lines as the copies of A and of the packed
// weights together.
template <int BITS, int MB, int NB, int WM, int WN, int STAGES, int SE, int GRP>
__global__ __launch_bounds__(WM* WN* kWave, 2) void qmmh_kernel(const QmmHalfArgs a) {
    constexpr bool G32 = GRP == 32;
    constexpr bool B8 = BITS == 8;
    constexpr float CENTRE = B8 ? 128.0f : 8.0f;  // the operand's codes are code - CENTRE
    static_assert(NB == 2, "a pair is two column blocks");
    constexpr int BM = WM * MB * 32;
    constexpr int BN = WN * NB * 32;
    constexpr int NWAVE = WM * WN;
    constexpr int A_STAGE = (BM / 32) * 4096;
    constexpr int QB = B8 ? 1 : 2;           // blocks of packed weights per stage
    constexpr int B_ROW = QB * 8 * BITS;     // bytes of a weight row per stage
    constexpr int B_BUFS = B8 ? STAGES : 2;
    constexpr int B_STAGE = BN * B_ROW;      // packed codes of QB 64-code blocks
    constexpr int A_BLOCKS = (BM / 32) * 4;  // 1 KiB fragments of A per stage
    constexpr int PPR = B_ROW / 16;          // 16-byte pieces of a row per stage
    constexpr int RPI = kWave / PPR;         // rows a copy instruction covers
    constexpr int NBC = B_STAGE / 1024 / NWAVE;  // B copies a wavefront issues per stage
    static_assert(A_BLOCKS % NWAVE == 0, "A fragments must divide among the wavefronts");
    static_assert(B_STAGE % (1024 * NWAVE) == 0 && NBC >= 1, "weight pieces must divide among the wavefronts");
    constexpr bool XS_LDS = !B8 && MB >= 3;  // the sums of x of a quad go through LDS
    constexpr int NX = (BM / 32 + NWAVE - 1) / NWAVE;  // copies of them a wavefront issues
    constexpr int NA = A_BLOCKS / NWAVE;  // A copies a wavefront issues per block
    constexpr bool WHOLE = MB == 1;                     // a block at a time (whole)
    constexpr int DEPTH = WHOLE ? STAGES - 1 : STAGES;  // blocks requested ahead of the loop
    // Behind the barrier of block g the copies of A's block g + STAGES are issued.  BITS 4: and, in a stage's first block, those of B's
    // stage after the next, two blocks before its codes are read; BITS 8: and B's block g + STAGES.  WHOLE: ahead of the barrier of
    // block g those of A's (and BITS 8's) block g + STAGES - 1 and, in a stage's first block, of BITS 4's next stage.  still_out: the
    // copies that may be on their way at the barrier of block Q of a quad: A of block g + 1 has to have landed and with it the codes
    // that are read up to the next barrier.
    static_assert(STAGES == 2 || STAGES == 3, "waits are counted for two or three stages");
    auto still_out = [=](int q) constexpr {
        return B8 ? (STAGES - 2) * (NA + NBC) : (STAGES - 2) * NA + ((q & 1) != WHOLE ? NBC : 0) + (XS_LDS && q == 1 ? NX : 0);
    };

    extern __shared__ __align__(16) uint8_t lds[];
    uint8_t* const abuf = lds;                     // [STAGES][A_STAGE]
    uint8_t* const bbuf = lds + STAGES * A_STAGE;  // [B_BUFS][B_STAGE]
    uint16_t* const sbuf = reinterpret_cast<uint16_t*>(bbuf + B_BUFS * B_STAGE);  // [scales, biases][BN][SE]
    // the same as LDS byte addresses: the copy instructions take theirs from a scalar register, and plain integer
    // arithmetic keeps it on the scalar unit (a pointer would be converted, null check included, per copy)
    const uint32_t abuf_at = __builtin_amdgcn_readfirstlane(lds_offset(lds));
    const uint32_t bbuf_at = abuf_at + STAGES * A_STAGE;

    const int row_bands = __builtin_amdgcn_readfirstlane(a.chunks ? *a.nchunks : a.tiles_m);
    const QmmTileAt at = qmmh_tile_at(a.seg, a.nseg, row_bands, (int)blockIdx.x);
    if (at.seg < 0) return;
    const int seg = __builtin_amdgcn_readfirstlane(at.seg);
    const int id = at.id, units = __builtin_amdgcn_readfirstlane(at.units);
    // tiles in groups of a.group_m row bands, column unit by column unit inside a group: the tiles an XCD works on at a
    // time then cover a patch of the output that is about as tall as it is wide in bytes read
    const int group = __builtin_amdgcn_readfirstlane(id / (a.group_m * units));
    const int in_group = id - group * a.group_m * units;
    const int bands = min(a.group_m, row_bands - group * a.group_m);
    const int unit = __builtin_amdgcn_readfirstlane(in_group / bands);
    const int tm = __builtin_amdgcn_readfirstlane(group * a.group_m + in_group - unit * bands);
    // shares of K from the last to the first, which then mostly is the one to add them up and still holds its own
    const int turns = __builtin_amdgcn_readfirstlane(unit / a.seg[seg].strips), split = a.seg[seg].ksplit - 1 - turns;
    const int tn = __builtin_amdgcn_readfirstlane(unit - turns * a.seg[seg].strips);
    float* const partial = a.seg[seg].partial;  // null: this workgroup's sums are whole
    uint32_t* const tickets = a.seg[seg].tickets;  // not null: partial sums are added here
    const bool pair = a.pair != 0;  // gate: seg[0], up: seg[1]

    const int tid = threadIdx.x;
    const int lane = tid & (kWave - 1);
    const int wave = __builtin_amdgcn_readfirstlane(tid / kWave);
    const int wave_m = wave / WN;
    const int wave_n = wave % WN;
    const int j = lane & 31;
    const int h = lane >> 5;

    const int K = a.K, N = a.seg[seg].N;
    const int Gall = K / 64;
    const int gb = __builtin_amdgcn_readfirstlane(split * a.seg[seg].gsplit);  // first block of K this workgroup multiplies (a multiple of 4)
    const int G = __builtin_amdgcn_readfirstlane(min(Gall, gb + a.seg[seg].gsplit));  // one past its last block
    const int G4 = (Gall + 3) / 4;
    const int ksteps = K / 16;
    const int sb_per_row = G32 ? Gall * 2 : Gall / a.gs_blocks;
    const int64_t words_per_row = (int64_t)K * BITS / 32;
    // a pointer picked or computed per workgroup, back on the scalar unit
    auto uniform = [](auto* p) {
        const uint64_t u = reinterpret_cast<uint64_t>(p);
        const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)u), hi = __builtin_amdgcn_readfirstlane((uint32_t)(u >> 32));
        return reinterpret_cast<decltype(p)>((uint64_t)hi << 32 | lo);
    };
    int m0 = tm * BM, mend = a.M;  // rows [m0, min(mend, m0 + BM)) of the fragments
    int64_t row1 = 0, row2 = 0;    // first weight row of the slab (PAIR: of either matrix)
    if (a.chunks) {
        const RouteChunk ch = a.chunks[tm];
        m0 = __builtin_amdgcn_readfirstlane(ch.first);
        mend = m0 + __builtin_amdgcn_readfirstlane(ch.count);
        const int64_t base = (int64_t)__builtin_amdgcn_readfirstlane(ch.expert) * a.expert_rows;
        row1 = base + a.row_base;
        row2 = base + a.row_base2;
    }
    const int n0 = tn * (pair ? BN / 2 : BN);
    // operands of column block 0 and 1 of the wavefronts' tiles
    const uint32_t* const w1 = uniform(a.seg[seg].w + row1 * words_per_row);
    const uint32_t* const w2 = uniform(pair ? a.seg[1].w + row2 * words_per_row : w1);
    const uint16_t* const sb1[2] = {uniform(a.seg[seg].s + row1 * sb_per_row), uniform(a.seg[seg].b + row1 * sb_per_row)};
    const uint16_t* const sb2[2] = {uniform(pair ? a.seg[1].s + row2 * sb_per_row : sb1[0]),
                                    uniform(pair ? a.seg[1].b + row2 * sb_per_row : sb1[1])};
    // weight row of column block nb, lane column c, for the wavefront column wn
    auto weight_row = [&](int wn, int nb, int c) { return min(pair ? n0 + wn * 32 + c : n0 + (wn * NB + nb) * 32 + c, N - 1); };

    // The tile's packed rows in 16-byte pieces: copy c of this wavefront fills 1 KiB, RPI rows of a stage, row r at r * B_ROW
    // bytes, its piece p at slot p ^ turn(r).  (Rows past N repeat the last row, pieces past K the last piece; a tile spans
    // well under 4 GiB, so the lane part fits 32 bits.  The RPI rows belong to one column block, hence to one matrix.)
    auto turn = [](int r) { return (r >> 2) & 3; };
    const int64_t first_row = (int64_t)min(n0, N - 1) * words_per_row;
    const uint32_t* const wtile1 = uniform(w1 + first_row);
    const uint32_t* const wtile2 = uniform(w2 + first_row);
    const uint32_t row_bytes = (uint32_t)(words_per_row * 4);
    uint32_t wrow[NBC], wpiece[NBC];
#pragma unroll
    for (int c = 0; c < NBC; c++) {
        const int r = (c * NWAVE + wave) * RPI + lane / PPR;  // row of the tile: column block r / 32
        wrow[c] = (uint32_t)(weight_row((r >> 5) / NB, (r >> 5) % NB, r & 31) - min(n0, N - 1)) * row_bytes;
        wpiece[c] = (uint32_t)((lane % PPR) ^ turn(r)) * 16u;
    }
    // copy c of stage st (64-code blocks QB * st ..) into buffer `buf`
    auto issue_b = [&](int c, int st, int buf) __attribute__((always_inline)) {
        const uint32_t in_row = min((uint32_t)(st * B_ROW) + wpiece[c], row_bytes - 16u);
        const int block = (c * NWAVE + wave) * RPI >> 5;
        copy16_to_lds((block & 1) ? wtile2 : wtile1, wrow[c] + in_row, bbuf_at + (uint32_t)(buf * B_STAGE + (c * NWAVE + wave) * 1024));
    };
    // copy c of A's block g
    auto issue_a1 = [&](int c, int g, int stage) __attribute__((always_inline)) {
        const int blk = wave + c * NWAVE;
        int mblk = m0 / 32 + (blk >> 2);
        mblk = mblk < a.mblks ? mblk : a.mblks - 1;  // past the end: any valid rows, never stored
        const uint16_t* src = a.xf + ((int64_t)mblk * ksteps + g * 4 + (blk & 3)) * 512;
        copy16_to_lds(src, (uint32_t)lane * 16u, abuf_at + (uint32_t)(stage * A_STAGE + blk * 1024));
    };
    const uint32_t mask_s = opaque_s(kMaskH);
    const uint32_t magic_v = opaque_v(kMagicH);
    // the first blocks are on their way while the prologue scans the scale rows
    if constexpr (!B8)
#pragma unroll
        for (int st = 0; st < (WHOLE ? 1 : 2); st++)
#pragma unroll
            for (int c = 0; c < NBC; c++) issue_b(c, min(gb / QB + st, (Gall - 1) / QB), st);
#pragma unroll
    for (int d = 0; d < DEPTH; d++) {
#pragma unroll
        for (int c = 0; c < NA; c++) issue_a1(c, gb + d < G ? gb + d : G - 1, d);
        if constexpr (B8)
#pragma unroll
            for (int c = 0; c < NBC; c++) issue_b(c, gb + d < G ? gb + d : G - 1, d);
    }

    // A row of scales (or biases) in pieces of eight elements.  Eight lanes share a row: a load touches eight lines.
    const uint32_t sb_total = (uint32_t)N * (uint32_t)sb_per_row;
    const int per_quad = G32 ? 8 : 4 / a.gs_blocks;                       // elements of a quad of four 64-code blocks
    const int first = gb / 4 * per_quad, last = min((G + 3) / 4 * per_quad, sb_per_row);  // of this workgroup's range of K
    auto sb_row = [&](int r) { return (uint32_t)weight_row((r >> 5) / NB, (r >> 5) % NB, r & 31) * (uint32_t)sb_per_row; };
    constexpr int THREADS = NWAVE * kWave;

    // Segment n of the scales and biases: SE elements of each row from first + n * SE on.  A thread loads its pieces (whose rows
    // lie in one matrix or, eight elements a segment, in two) and stores them later.
    constexpr int PPS = SE / 8;  // pieces of a row
    constexpr int NP = 2 * BN * PPS / THREADS;
    static_assert(2 * BN * PPS % THREADS == 0 && NP >= 1 && THREADS % kWave == 0, "pieces must divide among the threads");
    const int quads = G32 ? SE / 8 : a.gs_blocks == 1 ? SE / 4 : SE / 2;  // of a segment
    // (the thread's number is hidden from the compiler, which would keep every piece's address in registers)
    auto piece_off = [&](int i, int n, bool& bias, bool& second) __attribute__((always_inline)) {
        int t = tid;
        asm volatile("" : "+v"(t));
        const int at = i * THREADS + t, r = at / PPS % BN;
        bias = i * THREADS >= BN * PPS || ((i + 1) * THREADS > BN * PPS && at >= BN * PPS);
        second = (r >> 5) % NB != 0;
        return sb_row(r) + (uint32_t)(first + n * SE + at % PPS * 8);
    };
    auto load_segment = [&](auto tiny, int n, uint4 (&to)[NP]) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < NP; i++) {
            bool bias, second;
            const uint32_t off = piece_off(i, n, bias, second);
            to[i] = load_eight<decltype(tiny)::value>(bias ? (second ? sb2[1] : sb1[1]) : second ? sb2[0] : sb1[0], off, sb_total);
        }
    };
    auto store_segment = [&](int n, const uint4 (&from)[NP]) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < NP; i++) {
            bool bias, second;
            const uint32_t off = piece_off(i, n, bias, second);
            *reinterpret_cast<uint4*>(sbuf + (i * THREADS + tid) * 8) = moved_down(from[i], off, sb_total);
        }
    };
    uint4 piece[NP];

    // Ahead of the loop: the first segment, and the power of two that brings a row's largest scale (of this workgroup's range of K)
    // into [2^10, 2^11).  Everything is asked for before anything is waited for.
    float col_up[NB];
    auto scan = [&](auto tiny) __attribute__((always_inline)) {
        constexpr int ROWS = BN * 8 / THREADS;  // of a thread
        static_assert(BN * 8 % THREADS == 0, "rows of scales must divide among the threads");
        uint4 v[ROWS];
        uint32_t mag[ROWS];
        auto at = [&](int i, int e, const uint16_t*& base) {
            const int r = (i * THREADS + tid) >> 3;
            base = (r >> 5) % NB ? sb2[0] : sb1[0];
            return sb_row(r) + (uint32_t)e;
        };
        for (int e = first + (tid & 7) * 8, more = first; more < last; e += 64, more += 64) {
#pragma unroll
            for (int i = 0; i < ROWS; i++) {
                const uint16_t* base;
                const uint32_t off = at(i, e, base);
                v[i] = load_eight<decltype(tiny)::value>(base, off, sb_total);
            }
            if (more == first) {
#pragma unroll
                for (int i = 0; i < ROWS; i++) mag[i] = 0;
                load_segment(tiny, 0, piece);
            }
            const int n = last - e;  // elements that count
#pragma unroll
            for (int i = 0; i < ROWS; i++) {
                const uint16_t* base;
                const uint32_t off = at(i, e, base);
                v[i] = moved_down(v[i], off, sb_total);
                const uint32_t w[4] = {v[i].x, v[i].y, v[i].z, v[i].w};
                uint32_t most = 0;
#pragma unroll
                for (int c = 0; c < 4; c++) most = max_u16x2(most, w[c] & (n > 2 * c + 1 ? 0x7fff7fffu : n > 2 * c ? 0x7fffu : 0u));
                uint32_t one = max(most & 0xffffu, most >> 16);
                if (one >= 0x7f80u) {  // inf and NaN do not set the scale
                    one = 0;
#pragma nounroll
                    for (int c = 0; c < 8 && c < n; c++) {
                        const uint32_t m = (c < 4 ? (c < 2 ? w[0] : w[1]) : c < 6 ? w[2] : w[3]) >> (c & 1) * 16 & 0x7fffu;
                        if (m < 0x7f80u) one = max(one, m);
                    }
                }
                mag[i] = max(mag[i], one);
            }
        }
        uint32_t* const mags = reinterpret_cast<uint32_t*>(sbuf);
#pragma unroll
        for (int i = 0; i < ROWS; i++) {
            mag[i] = max(mag[i], (uint32_t)__builtin_amdgcn_mov_dpp((int)mag[i], 0xb1, 0xf, 0xf, false));   // quad_perm 1 0 3 2
            mag[i] = max(mag[i], (uint32_t)__builtin_amdgcn_mov_dpp((int)mag[i], 0x4e, 0xf, 0xf, false));   // quad_perm 2 3 0 1
            mag[i] = max(mag[i], (uint32_t)__builtin_amdgcn_mov_dpp((int)mag[i], 0x141, 0xf, 0xf, false));  // eight lanes mirrored
            if ((tid & 7) == 0) mags[(i * THREADS + tid) >> 3] = mag[i];
        }
        __syncthreads();
#pragma unroll
        for (int nb = 0; nb < NB; nb++) col_up[nb] = pow2f(exponent_shift(mags[(wave_n * NB + nb) * 32 + j], 10));
        __syncthreads();
    };
    auto prologue = [&](auto tiny) __attribute__((always_inline)) {
        if constexpr (B8) {  // the scales stay fp32
#pragma unroll
            for (int nb = 0; nb < NB; nb++) col_up[nb] = 1.0f;
            load_segment(tiny, 0, piece);
        } else {
            scan(tiny);
        }
    };
    // The rows' factors wait in LDS for the epilogue, whose first loads they were, behind all of K and ahead of every store (2048 rows of 4096 /
    // 14336 937 -> 926 us, 777 rows of 8 bit 322 -> 318, 509 rows in groups of 32 359 -> 357; 40 layers of 66 to 2048 rows 0.7 % faster).
    constexpr bool RS_LDS = half_rows_in_lds(BITS, MB, NWAVE);
    static_assert(BM <= THREADS, "a row's factor a thread");
    float* const rbuf = reinterpret_cast<float*>(sbuf + 2 * BN * SE) + (XS_LDS ? BM / 32 * 256 : 0);
    [[maybe_unused]] float row_down = 0.0f;
    if constexpr (RS_LDS)
        if (tid < BM) row_down = a.rs[min(m0 + tid, a.mblks * 32 - 1)];
    if (sb_total < 8)
        prologue(std::true_type{});
    else
        prologue(std::false_type{});
    store_segment(0, piece);
    if constexpr (RS_LDS)
        if (tid < BM) rbuf[tid] = row_down;
    // A quad's scales (which 0) or biases (1) of this lane's rows: the bf16 bits of its four blocks in two words per column block
    // (groups of 32: this lane half's four of the quad's eight).
    const uint32_t half_sel = h ? 0x07060302u : 0x05040100u;
    const uint32_t sel_01 = a.gs_blocks == 1 ? 0x03020100u : 0x01000100u, sel_23 = a.gs_blocks == 1 ? 0x07060504u : 0x03020302u;
    uint2 s_cur[NB], s_nxt[NB], b_cur[NB];
    auto read_quad = [&](int which, int quad, uint2 (&dst)[NB]) __attribute__((always_inline)) {
#pragma unroll
        for (int nb = 0; nb < NB; nb++) {
            const uint16_t* const at = sbuf + ((which * BN + (wave_n * NB + nb) * 32 + j) * SE + quad * per_quad);
            if constexpr (G32) {
                const uint4 v = *reinterpret_cast<const uint4*>(at);
                dst[nb] = make_uint2(__builtin_amdgcn_perm(v.y, v.x, half_sel), __builtin_amdgcn_perm(v.w, v.z, half_sel));
            } else {  // (groups of 128: two elements, each for two blocks)
                const uint32_t lo = *reinterpret_cast<const uint32_t*>(at), hi = *reinterpret_cast<const uint32_t*>(at + per_quad - 2);
                dst[nb] = make_uint2(__builtin_amdgcn_perm(hi, lo, sel_01), __builtin_amdgcn_perm(hi, lo, sel_23));
            }
        }
    };
    // bf16 bits of block q (0..3) of a quad, as the high half of a word (= the fp32 value)
    auto quad_hi = [](const uint2& v, int q) {
        const uint32_t w = q < 2 ? v.x : v.y;
        return (q & 1) ? (w & 0xffff0000u) : (w << 16);
    };
    int quad_at = 0;  // place of the quad under way in its segment
    int segment = 0;
    // Sums of x: loaded a quad at a time, or, where registers are short, copied into LDS, a row block a copy
    // (several wavefronts the same one where there are fewer): 512 bytes a quad, groups of 32 1024.
    constexpr int XS_BLOCK = G32 ? 1024 : 512;
    const uint32_t xbuf_at = bbuf_at + B_BUFS * B_STAGE + 2 * BN * SE * 2;
    const uint8_t* const xbuf = reinterpret_cast<const uint8_t*>(sbuf) + 2 * BN * SE * 2;
    [[maybe_unused]] auto issue_xs = [&](int quad) __attribute__((always_inline)) {
#pragma unroll
        for (int c = 0; c < NX; c++) {
            const int blk = (wave + c * NWAVE) % (BM / 32), mblk = min(m0 / 32 + blk, a.mblks - 1);
            copy16_to_lds(reinterpret_cast<const uint8_t*>(a.xs) + ((int64_t)mblk * G4 + quad) * XS_BLOCK, (uint32_t)(G32 ? lane : lane & 31) * 16u,
                          xbuf_at + (uint32_t)(blk * 1024));
        }
    };
    [[maybe_unused]] uint32_t xsoff[MB];  // in 16-byte units
#pragma unroll
    for (int mb = 0; mb < MB; mb++) {
        const int mblk = min(m0 / 32 + wave_m * MB + mb, a.mblks - 1);
        xsoff[mb] = (uint32_t)mblk * (uint32_t)(G32 ? 2 * G4 : G4) * 32u + (G32 ? (uint32_t)h * 32u : 0u) + (uint32_t)j;
    }
    uint4 xs_cur[XS_LDS ? 1 : MB];
    auto load_xs = [&](int quad) {
#pragma unroll
        for (int mb = 0; mb < (XS_LDS ? 0 : MB); mb++) xs_cur[mb] = reinterpret_cast<const uint4*>(a.xs)[xsoff[mb] + (G32 ? 64 * quad : 32 * quad)];
    };

    f32x16_t out[MB][NB];
#pragma unroll
    for (int mb = 0; mb < MB; mb++)
#pragma unroll
        for (int nb = 0; nb < NB; nb++)
#pragma unroll
            for (int r = 0; r < 16; r++) out[mb][nb][r] = 0.0f;

    // Affine terms of a quad's blocks 0..qlast in one bf16 MFMA per output tile: k-slots (2q, 2q+1) carry
    // (Sx_hi, Sx_lo) of block q on the A side; lanes h=0 pair them with the bias, lanes h=1 with 8 * scale
    // (both times the row's power of two: exact); blocks past qlast (only at the end of K) contribute zeros.
    auto affine = [&](int qlast) __attribute__((always_inline)) {
        bf16x8_t bbf[NB], ebf[NB];
#pragma unroll
        for (int nb = 0; nb < NB; nb++) {
            uint32_t v[4], ve[4];
#pragma unroll
            for (int q = 0; q < 4; q++) {
                if (q <= qlast) {
                    const uint32_t eight = __float_as_uint(__uint_as_float(quad_hi(s_cur[nb], q)) * (CENTRE * col_up[nb])) >> 16;
                    const uint32_t bia = __float_as_uint(__uint_as_float(quad_hi(b_cur[nb], q)) * col_up[nb]) >> 16;
                    v[q] = dup16(!G32 && h ? eight : bia);
                    ve[q] = dup16(eight);
                } else {
                    v[q] = ve[q] = 0u;
                }
            }
            const uint4 u = {v[0], v[1], v[2], v[3]}, ue = {ve[0], ve[1], ve[2], ve[3]};
            bbf[nb] = __builtin_bit_cast(bf16x8_t, u);
            ebf[nb] = __builtin_bit_cast(bf16x8_t, ue);
        }
        if constexpr (XS_LDS) __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int mb = 0; mb < MB; mb++) {
            const uint4 sums = XS_LDS ? *reinterpret_cast<const uint4*>(xbuf + (wave_m * MB + mb) * 1024 + (G32 ? lane : j) * 16) : xs_cur[XS_LDS ? 0 : mb];
            const bf16x8_t aa = __builtin_bit_cast(bf16x8_t, sums);
#pragma unroll
            for (int nb = 0; nb < NB; nb++)
                out[mb][nb] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(aa, bbf[nb], out[mb][nb], 0, 0, 0);
            if constexpr (G32) {
#pragma unroll
                for (int nb = 0; nb < NB; nb++)
                    out[mb][nb] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(aa, ebf[nb], out[mb][nb], 0, 0, 0);
            }
            if constexpr (XS_LDS) __builtin_amdgcn_sched_barrier(0);
        }
    };

    // A 64-code block at a time; Q = g & 3 is static so that everything indexed by it stays in fixed registers.  Past the end of K the
    // last block is requested again.  Who asks for what, which barrier publishes it and which frees its place:
    //   copies of A and of the packed weights: see still_out;
    //   the segment of scales and biases after this one, in the last quad of a segment: ordinary loads at the start of block Q = 1, stored
    //     over the old segment ahead of that block's barrier.  The old one's last scales and biases have been read by every wavefront
    //     before the barrier of Q = 0 (or of the Q = 3 before it); the new ones are first read at Q = 3 (BITS 8: at the next Q = 0);
    //   a quad's sums of x: BITS 4 ordinary loads at Q = 1, or with XS_LDS copies behind the barrier of Q = 0, which has freed their
    //     place (the last quad's are read at the end of Q = 3) and which the barrier of Q = 2 publishes; BITS 8 ordinary loads at Q = 2
    //     (WHOLE: at Q = 1).
    // The compiler cannot count the copy instructions, so wherever it first uses a register of an ordinary load it waits until NOTHING is
    // outstanding, copies included.  A block with ordinary loads is therefore ordered: loads, MFMAs, first use of the loaded registers
    // (forced), and only then new copies - the forced wait then covers the loads, most of a block of MFMAs old, and the copies that the
    // barrier waits for anyway.
    // With two stages the stage of block g is g & 1, static like Q, and every LDS address of the loop is a constant; with three it is
    // carried along.
    constexpr bool STATIC_STAGE = STAGES == 2;
    int sa_carried = 0;  // LDS stage that holds block g
    // whether the quad of block g is the last of its segment, with more of K behind it
    auto refills = [&](int g) { return quad_at + 1 == quads && (g | 3) + 1 < G; };
    auto next_quad = [&] {
        if (++quad_at == quads) quad_at = 0, segment++;
    };
    // BITS 4: the loop as a pipeline of steps of 16 codes.  Step t of a block multiplies the fragments that step t - 1 has made
    // ready, while the words of step t + 1 are expanded and A's fragments of step t + 1 are read, both a few instructions at a
    // time between the MFMAs of one row block and the next: a wavefront then keeps matrix cores, vector unit and LDS busy by
    // itself, where expanding a whole block ahead of its MFMAs left the matrix cores to the one other wavefront of the SIMD.
    // The only barrier of a block is in the middle of its last step, behind MFMAs that need nothing of the next block.
    constexpr bool TWO_A = MB <= 3;  // A's next fragments in registers of their own; else over those just multiplied
    f16x8_t afr[WHOLE ? 4 : TWO_A ? 2 : 1][MB];
    uint32_t bfr[WHOLE ? 4 : 2][NB][4];
    uint4 cw[NB];               // the block's words of this lane
    f16x2_t s2[NB], m24[NB];    // its scale, brought into fp16 range (8 significant bits: exact), and -24 times it (10 bits)
    auto read_a = [&](int mb, int t, int stage) {
        afr[WHOLE ? t : TWO_A ? t & 1 : 0][mb] = *reinterpret_cast<const f16x8_t*>(abuf + stage * A_STAGE + (wave_m * MB + mb) * 4096 + t * 1024 + lane * 16);
    };
    // row (wave_n * NB + nb) * 32 + j, words 4h .. 4h+3, of block Q of a quad
    auto read_codes = [&](int q) {
#pragma unroll
        for (int nb = 0; nb < NB; nb++)
            cw[nb] = *reinterpret_cast<const uint4*>(bbuf + (q >> 1) * B_STAGE + ((wave_n * NB + nb) * 32 + j) * B_ROW + (((q % 2 * 2 + h) ^ turn(j)) * 16));
    };
    auto take_scale = [&](const uint2 (&from)[NB], int q) {
#pragma unroll
        for (int nb = 0; nb < NB; nb++) {
            const float sv = __uint_as_float(quad_hi(from[nb], q)) * col_up[nb], mv = sv * -24.0f;
            s2[nb] = f16x2_t{(_Float16)sv, (_Float16)sv};
            m24[nb] = f16x2_t{(_Float16)mv, (_Float16)mv};
        }
    };
    // pairs [from, to) of the NB * 4 of word t
    auto expand_some = [&](int t, int from, int to) __attribute__((always_inline)) {
#pragma unroll
        for (int i = from; i < to; i++) {
            const int nb = i >> 2;
            const uint32_t w = t == 0 ? cw[nb].x : t == 1 ? cw[nb].y : t == 2 ? cw[nb].z : cw[nb].w;
            uint32_t& to_reg = bfr[WHOLE ? t : t & 1][nb][i & 3];
            if ((i & 3) == 0) to_reg = expand_pair<0>(w, mask_s, magic_v, s2[nb], m24[nb]);
            if ((i & 3) == 1) to_reg = expand_pair<1>(w, mask_s, magic_v, s2[nb], m24[nb]);
            if ((i & 3) == 2) to_reg = expand_pair<2>(w, mask_s, magic_v, s2[nb], m24[nb]);
            if ((i & 3) == 3) to_reg = expand_pair<3>(w, mask_s, magic_v, s2[nb], m24[nb]);
        }
    };
    auto block = [&](auto q_tag, int g) __attribute__((always_inline)) {
        constexpr int Q = decltype(q_tag)::value;
        const int sa = STATIC_STAGE ? Q % STAGES : sa_carried;
        const int sa_next = sa == STAGES - 1 ? 0 : sa + 1;
        constexpr int PRE = MB / 2;  // row blocks of the last step ahead of the barrier
        constexpr int PAIRS = NB * 4;
        const bool refill = Q == 1 && refills(g);
        if constexpr (Q == 0) read_quad(1, quad_at, b_cur);
        if constexpr (Q == 1) {
            if (refill) load_segment(std::false_type{}, segment + 1, piece);
            if constexpr (!XS_LDS) load_xs(g >> 2);
            __builtin_amdgcn_sched_barrier(0);
        }
        if constexpr (Q == 3) read_quad(0, quad_at + 1 == quads ? 0 : quad_at + 1, s_nxt);  // (behind the end of K: anything)
#pragma unroll
        for (int t = 0; t < 4; t++) {
            const int tn = (t + 1) & 3;  // the step that is made ready
            if (t == 3) {  // the last word of this block is expanded
                read_codes((Q + 1) & 3);
                if (Q == 3) take_scale(s_nxt, 0); else take_scale(s_cur, Q + 1);
            }
#pragma unroll
            for (int mb = 0; mb < MB; mb++) {
                if (t == 3 && mb == PRE) {
                    // The ordinary loads of block 1 are first used here, ahead of new copies: the compiler, which cannot count
                    // the copies, waits for everything.
                    if constexpr (Q == 1) {
                        if (refill) store_segment(segment + 1, piece);
#pragma unroll
                        for (int m = 0; m < (XS_LDS ? 0 : MB); m++)
                            asm volatile("" : "+v"(xs_cur[m].x), "+v"(xs_cur[m].y), "+v"(xs_cur[m].z), "+v"(xs_cur[m].w));
                    }
                    // What the next block needs has landed once only newer copies are outstanding, and every read of this block
                    // has returned.  A bare s_barrier on purpose: __syncthreads() carries a workgroup fence, for which the
                    // compiler drains ALL outstanding copies into LDS.
                    __builtin_amdgcn_sched_barrier(0);
                    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(still_out(Q)) : "memory");
                    __builtin_amdgcn_s_barrier();
                    asm volatile("" ::: "memory");
                    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                    for (int m = 0; m < PRE; m++) read_a(m, 0, sa_next);
                }
                const bool reads = t < 3 || mb >= PRE;
                if (TWO_A && reads) read_a(mb, tn, t == 3 ? sa_next : sa);
#pragma unroll
                for (int nb = 0; nb < NB; nb++)
                    out[mb][nb] = __builtin_amdgcn_mfma_f32_32x32x16_f16(afr[TWO_A ? t & 1 : 0][mb], __builtin_bit_cast(f16x8_t, make_uint4(bfr[t & 1][nb][0], bfr[t & 1][nb][1], bfr[t & 1][nb][2], bfr[t & 1][nb][3])),
                                                                         out[mb][nb], 0, 0, 0);
                if (!TWO_A && reads) read_a(mb, tn, t == 3 ? sa_next : sa);
                expand_some(tn, mb * PAIRS / MB, (mb + 1) * PAIRS / MB);
                if (t == 3 && mb >= PRE) {
                    constexpr int COPIES = NA + ((Q & 1) == 0 ? NBC : 0), OVER = MB - PRE;
#pragma unroll
                    for (int c = (mb - PRE) * COPIES / OVER; c < (mb - PRE + 1) * COPIES / OVER; c++) {
                        if (c < NA)
                            issue_a1(c, min(g + STAGES, G - 1), sa);
                        else
                            issue_b(c - NA, min(g / QB + 2, (Gall - 1) / QB), Q >> 1);
                    }
                    // (the last quad's sums have been read before this barrier)
                    if (XS_LDS && Q == 0 && mb == MB - 1) issue_xs(g >> 2);
                }
                __builtin_amdgcn_sched_barrier(0);
            }
        }
        if constexpr (Q == 3) {
            affine(3);
#pragma unroll
            for (int nb = 0; nb < NB; nb++) s_cur[nb] = s_nxt[nb];
            next_quad();
        }
        sa_carried = sa_next;
    };
    // BITS 8: units of the MFMAs of a row block and group, into partial sums of their own.  While a unit is multiplied the sums of the
    // unit before it are scaled; in a block's last row block, behind the barrier, each step's fragments of B are replaced by the next
    // block's as soon as they have been multiplied, and A's always by the next row block's.  A quad ends with its sums scaled.
    constexpr int GROUPS = G32 ? 2 : 1;  // of a block
    constexpr int UNITS = MB * GROUPS, STEPS = 4 / GROUPS;
    f16x8_t a8[4], b8[NB][4];
    uint4 codes8[NB];  // of two steps
    constexpr int PARTS = G32 || WHOLE ? 1 : 2;  // (groups of 32 have no registers for a second unit's sums: scaled behind their own MFMAs)
    f32x16_t part[PARTS][NB];
    float scale[NB][GROUPS], scale_before[NB];  // of the block's groups; of the last group of the block before
    // (the compiler would move what it can of the work above a branch behind it, with everything that this work reads)
    auto pin8 = [&]() __attribute__((always_inline)) {
#pragma unroll
        for (int nb = 0; nb < NB; nb++) {
#pragma unroll
            for (int mb = 0; mb < MB; mb++) asm volatile("" : "+v"(out[mb][nb]));
#pragma unroll
            for (int t = 0; t < 4; t++) asm volatile("" : "+v"(b8[nb][t]));
        }
    };
    auto read_a8 = [&](int t, int mb, int stage) __attribute__((always_inline)) {
        a8[t] = *reinterpret_cast<const f16x8_t*>(abuf + stage * A_STAGE + (wave_m * MB + mb) * 4096 + t * 1024 + lane * 16);
    };
    // Row (wave_n * NB + nb) * 32 + j: the sixteen codes of steps 2 i and 2 i + 1, whole 16-byte pieces of 16 rows that lie in different
    // banks.  (Eight codes a read, one half of each piece: rows j and j + 16 met in the same banks; conflicts took
    // 13 % of a CU's cycles in gate and up of 777 rows, 6 % so.)
    auto read_codes8 = [&](int i, int stage) __attribute__((always_inline)) {
        const uint8_t* const at = bbuf + (stage * B_STAGE + (wave_n * NB * 32 + j) * B_ROW + (((2 * i + h) ^ turn(j)) * 16));
#pragma unroll
        for (int nb = 0; nb < NB; nb++) codes8[nb] = *reinterpret_cast<const uint4*>(at + nb * 32 * B_ROW);
    };
    auto expand8 = [&](int t) __attribute__((always_inline)) {
#pragma unroll
        for (int nb = 0; nb < NB; nb++) b8[nb][t] = expand_bytes(t & 1 ? make_uint2(codes8[nb].z, codes8[nb].w) : make_uint2(codes8[nb].x, codes8[nb].y));
    };
    auto take_scales8 = [&](int q) __attribute__((always_inline)) {  // of block q of a quad
#pragma unroll
        for (int nb = 0; nb < NB; nb++) {
            const uint32_t sv = quad_hi(s_cur[nb], q);
            if constexpr (G32) {  // the lane halves hold the two groups' scales
                const auto both = __builtin_amdgcn_permlane32_swap(sv, sv, false, false);
                scale[nb][0] = __uint_as_float(both[0]);
                scale[nb][1] = __uint_as_float(both[1]);
            } else {
                scale[nb][0] = __uint_as_float(sv);
            }
        }
    };
    // registers [from, to) of the sums of the unit before unit u of block Q of a quad
    auto scale_part = [&](auto q_tag, int u, int from, int to) __attribute__((always_inline)) {
        constexpr int Q = decltype(q_tag)::value;
        const int last = u == 0 ? UNITS - 1 : u - 1;
#pragma unroll
        for (int nb = 0; nb < NB; nb++)
#pragma unroll
            for (int r = from; r < to; r++)
                out[last / GROUPS][nb][r] = __builtin_fmaf(u == 0 ? scale_before[nb] : scale[nb][last % GROUPS], part[(Q * UNITS + u + 1) % PARTS][nb][r],
                                                           out[last / GROUPS][nb][r]);
    };
    [[maybe_unused]] auto block8 = [&](auto q_tag, int g) __attribute__((always_inline)) {
        constexpr int Q = decltype(q_tag)::value;
        const int sa = sa_carried, sa_next = sa == STAGES - 1 ? 0 : sa + 1;
        const bool refill = Q == 1 && refills(g);
        if constexpr (Q == 0) {
            read_quad(0, quad_at, s_cur);
            read_quad(1, quad_at, b_cur);
        }
        if constexpr (Q == 1) pin8();
        if (refill) load_segment(std::false_type{}, segment + 1, piece);
        if constexpr (Q == 2) load_xs(g >> 2);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int u = 0; u < UNITS; u++) {
            const int mb = u / GROUPS;
            const bool last_mb = mb == MB - 1;
            if (u == (MB - 1) * GROUPS) {  // (as in BITS 4's)
                if constexpr (Q == 1) pin8();
                if (refill) store_segment(segment + 1, piece);
                if constexpr (Q == 2) {
#pragma unroll
                    for (int m = 0; m < MB; m++)
                        asm volatile("" : "+v"(xs_cur[m].x), "+v"(xs_cur[m].y), "+v"(xs_cur[m].z), "+v"(xs_cur[m].w));
                }
                __builtin_amdgcn_sched_barrier(0);
                asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(still_out(Q)) : "memory");
                __builtin_amdgcn_s_barrier();
                asm volatile("" ::: "memory");
                __builtin_amdgcn_sched_barrier(0);
            }
#pragma unroll
            for (int step = 0; step < STEPS; step++) {
                const int t = u % GROUPS * STEPS + step;
#pragma unroll
                for (int nb = 0; nb < NB; nb++)
                    part[(Q * UNITS + u) % PARTS][nb] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a8[t], b8[nb][t], step ? part[(Q * UNITS + u) % PARTS][nb] : f32x16_t{}, 0, 0, 0);
                read_a8(t, last_mb ? 0 : mb + 1, last_mb ? sa_next : sa);
                if (PARTS == 2 && (Q > 0 || u > 0)) scale_part(q_tag, u, step * 16 / STEPS, (step + 1) * 16 / STEPS);
                if (u == 0 && step == STEPS - 1) take_scales8(Q);
                if (last_mb) {
                    if (t > 0) expand8(t - 1);
                    if (t % 2 == 0) read_codes8(t / 2, sa_next);
#pragma unroll
                    for (int c = t * (NA + NBC) / 4; c < (t + 1) * (NA + NBC) / 4; c++) {
                        if (c < NA)
                            issue_a1(c, min(g + STAGES, G - 1), sa);
                        else
                            issue_b(c - NA, min(g + STAGES, G - 1), sa);
                    }
                }
                __builtin_amdgcn_sched_barrier(0);
            }
            if (PARTS == 1) {
                scale_part(q_tag, u + 1, 0, 16);
                __builtin_amdgcn_sched_barrier(0);
            }
        }
        expand8(3);
        if constexpr (Q == 3) {
            if (PARTS == 2) scale_part(q_tag, UNITS, 0, 16);
            affine(3);
            next_quad();
        } else {
#pragma unroll
            for (int nb = 0; nb < NB; nb++) scale_before[nb] = scale[nb][GROUPS - 1];
        }
        __builtin_amdgcn_sched_barrier(0);
        sa_carried = sa_next;
    };
    // 32 rows a wavefront: a block's codes are expanded, then multiplied (BITS 8: then its sums scaled), while the other wavefronts of
    // the SIMD fill the matrix cores.  With two MFMAs a step the pipelines above have too little to hide LDS latency behind.  us,
    // pipeline -> here.  BITS 4, 32 x 256 tiles: 413 x 4096 x 3328 46.0 -> 39.7, 413 x 1024 x 3328 17.4 -> 15.7, in groups of 32 300 x
    // 2048 x 3328 28.6 -> 25.2; 512 tokens through 128 experts (2816 / 704) gate|up 121.8 -> 114.6, down 74.7 -> 72.4; level at three
    // tiles a CU.  BITS 8: block8 takes 196 registers for 64 x 128 tiles (groups of 32 178), which leaves two wavefronts a SIMD where
    // LDS has room for three; here 136 (164): 777 x 2560 x 3072 63.6 -> 53.4, the experts 160.9 -> 151.5 and 100.3 -> 85.7, in groups
    // of 32 182.5 -> 179.1 and 105.7 -> 89.7; 32 x 256 tiles 777 x 2048 x 2560 29.0 -> 28.1, 777 x 2560 x 20480 188 -> 172.
    // The copies of block g + STAGES - 1 go to the stage that was last read in block g - 1, BITS 4's next stage of B likewise; in
    // block 1 they follow the first use of its ordinary loads.
    [[maybe_unused]] auto whole = [&](auto q_tag, int g) __attribute__((always_inline)) {
        constexpr int Q = decltype(q_tag)::value;
        const int sa = sa_carried, st2 = sa == 0 ? STAGES - 1 : sa - 1, g2 = min(g + STAGES - 1, G - 1);
        const bool refill = Q == 1 && refills(g);
        auto request = [&]() __attribute__((always_inline)) {
#pragma unroll
            for (int c = 0; c < NA; c++) issue_a1(c, g2, st2);
            if constexpr (B8 || Q % 2 == 0)
#pragma unroll
                for (int c = 0; c < NBC; c++) B8 ? issue_b(c, g2, st2) : issue_b(c, min(g / QB + 1, (Gall - 1) / QB), (Q >> 1) ^ 1);
        };
        if constexpr (Q == 0) {
            if constexpr (B8) read_quad(0, quad_at, s_cur);
            read_quad(1, quad_at, b_cur);
        }
        if constexpr (Q == 3 && !B8) read_quad(0, quad_at + 1 == quads ? 0 : quad_at + 1, s_nxt);  // (behind the end of K: anything)
        if constexpr (Q == 1) {
            if (refill) load_segment(std::false_type{}, segment + 1, piece);
            load_xs(g >> 2);
        } else {
            request();
        }
        if constexpr (B8) {
#pragma unroll
            for (int t = 0; t < 4; t++) {
                if (t % 2 == 0) read_codes8(t / 2, sa);
                expand8(t);
            }
            take_scales8(Q);
#pragma unroll
            for (int t = 0; t < 4; t++) read_a8(t, 0, sa);
#pragma unroll
            for (int u = 0; u < GROUPS; u++) {
#pragma unroll
                for (int step = 0; step < STEPS; step++)
#pragma unroll
                    for (int nb = 0; nb < NB; nb++)
                        part[0][nb] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a8[u * STEPS + step], b8[nb][u * STEPS + step], step ? part[0][nb] : f32x16_t{}, 0, 0, 0);
                scale_part(q_tag, u + 1, 0, 16);
            }
        } else {
            read_codes(Q);
            take_scale(s_cur, Q);
#pragma unroll
            for (int t = 0; t < 4; t++) read_a(0, t, sa);
#pragma unroll
            for (int t = 0; t < 4; t++) {
                expand_some(t, 0, NB * 4);
#pragma unroll
                for (int nb = 0; nb < NB; nb++)
                    out[0][nb] = __builtin_amdgcn_mfma_f32_32x32x16_f16(afr[t][0], __builtin_bit_cast(f16x8_t, make_uint4(bfr[t][nb][0], bfr[t][nb][1], bfr[t][nb][2], bfr[t][nb][3])),
                                                                        out[0][nb], 0, 0, 0);
            }
        }
        if constexpr (Q == 1) {
            __builtin_amdgcn_sched_barrier(0);
            if (refill) store_segment(segment + 1, piece);
            asm volatile("" : "+v"(xs_cur[0].x), "+v"(xs_cur[0].y), "+v"(xs_cur[0].z), "+v"(xs_cur[0].w));
            __builtin_amdgcn_sched_barrier(0);
            request();
        }
        if constexpr (Q == 3) {
            affine(3);
            if constexpr (!B8)
#pragma unroll
                for (int nb = 0; nb < NB; nb++) s_cur[nb] = s_nxt[nb];
            next_quad();
        }
        // (or the compiler moves work behind the next branch, and what it reads stays in registers until there: BITS 8's partial sums)
#pragma unroll
        for (int nb = 0; nb < NB; nb++) asm volatile("" : "+v"(out[0][nb]));
        sa_carried = sa == STAGES - 1 ? 0 : sa + 1;
        asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(still_out(Q)) : "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
    };
    // blocks 0 .. DEPTH-1 were requested before the scan of the scale rows (any wait of the compiler's for the loads since then has
    // drained those copies too)
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"((DEPTH - 1) * (B8 ? NA + NBC : NA)) : "memory");  // block 0 has landed
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    auto run = [&](auto q_tag, int g) __attribute__((always_inline)) {
        if constexpr (WHOLE) whole(q_tag, g); else if constexpr (B8) block8(q_tag, g); else block(q_tag, g);
    };
    if constexpr (B8 && !WHOLE) {
#pragma unroll
        for (int t = 0; t < 4; t++) {
            if (t % 2 == 0) read_codes8(t / 2, 0);
            expand8(t);
            read_a8(t, 0, 0);
        }
    } else if constexpr (!B8) {
        read_quad(0, 0, s_cur);
        if constexpr (!WHOLE) {
            read_codes(0);
            take_scale(s_cur, 0);
#pragma unroll
            for (int mb = 0; mb < MB; mb++) read_a(mb, 0, 0);
            expand_some(0, 0, NB * 4);
        }
    }
    int g = gb;
    for (; g + 4 <= G; g += 4) {
        run(std::integral_constant<int, 0>{}, g);
        run(std::integral_constant<int, 1>{}, g + 1);
        run(std::integral_constant<int, 2>{}, g + 2);
        run(std::integral_constant<int, 3>{}, g + 3);
    }
    g = __builtin_amdgcn_readfirstlane(g);
    if (g < G) {  // K ends inside a quad
        run(std::integral_constant<int, 0>{}, g);
        if constexpr (B8 && PARTS == 2)
            if (g + 1 == G) scale_part(std::integral_constant<int, 0>{}, UNITS, 0, 16);
        if (g + 1 < G) run(std::integral_constant<int, 1>{}, g + 1);
        if constexpr (B8 && PARTS == 2)
            if (g + 2 == G) scale_part(std::integral_constant<int, 1>{}, UNITS, 0, 16);
        if (g + 2 < G) run(std::integral_constant<int, 2>{}, g + 2);
        if constexpr (B8 && PARTS == 2)
            if (g + 3 == G) scale_part(std::integral_constant<int, 2>{}, UNITS, 0, 16);
        if constexpr (XS_LDS) {  // its sums are asked for in its first block, and may be on their way
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
            __builtin_amdgcn_s_barrier();
            asm volatile("" ::: "memory");
        } else if (g + (B8 && !WHOLE ? 2 : 1) >= G) {
            load_xs(g >> 2);
        }
        affine(G - 1 - g);
    }
    // the copies requested past the end of K must not outlive the wavefront's use of LDS
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");

    // D layout of v_mfma_f32_32x32x*: lane (j, h), register r -> row 8*(r/4) + 4*h + r%4, column j: a lane holds
    // single elements of 16 rows, and storing them as they lie means 2-byte stores to 64-byte pieces of rows
    // (measured: a third of a tile's time).  Each 32-row block of the wavefront's tile, scaled by the two inverse powers of two
    // (exact, whatever the order; that of the column belongs to the share of K, whose scales it comes from), therefore goes through a
    // staging area in LDS that belongs to the wavefront (the stages are free: every copy has landed, every read of
    // the loop has returned, and the barrier says so for all wavefronts) and leaves it row-major, eight consecutive columns per lane: 16-byte bf16
    // stores, whole 128-byte lines per eight lanes.
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    {
        const float col_down[2] = {1.0f / col_up[0], 1.0f / col_up[1]};
#pragma unroll
        for (int mb = 0; mb < MB; mb++) {
            const int in_tile = (wave_m * MB + mb) * 32;
#pragma unroll
            for (int q = 0; q < 4; q++) {
                const int r = in_tile + 4 * h + 8 * q, m = m0 + r;  // m < mblks * 32 unless the whole block lies past the last row
                float4 down = make_float4(0.f, 0.f, 0.f, 0.f);
                if constexpr (RS_LDS)
                    down = *reinterpret_cast<const float4*>(rbuf + r);
                else if (m < a.mblks * 32)
                    down = *reinterpret_cast<const float4*>(a.rs + m);
#pragma unroll
                for (int nb = 0; nb < NB; nb++) {
                    out[mb][nb][4 * q] = out[mb][nb][4 * q] * down.x * col_down[nb];
                    out[mb][nb][4 * q + 1] = out[mb][nb][4 * q + 1] * down.y * col_down[nb];
                    out[mb][nb][4 * q + 2] = out[mb][nb][4 * q + 2] * down.z * col_down[nb];
                    out[mb][nb][4 * q + 3] = out[mb][nb][4 * q + 3] * down.w * col_down[nb];
                }
            }
        }
    }
    if (tickets) {
        // Shares of K (aq_share_sum.h): the sums of 32 x 32 blocks as the accumulators hold them, [share][block row][block column,
        // gate then up][four accumulators][lane].
        const int cols = (N + 31) / 32, all_cols = pair ? 2 * cols : cols, shares = a.seg[seg].ksplit;
        const uint32_t share = (uint32_t)a.mblks * all_cols * 4096;
        auto of = [&](int s) { return partial_sums(uniform(partial + (int64_t)s * (share / 4)), share); };
        // block (mb, nb) of this wavefront's tile; past the last row or column: past the end
        auto block_at = [&](int mb, int nb) {
            const int br = m0 / 32 + wave_m * MB + mb, bc = pair ? n0 / 32 + wave_n : n0 / 32 + wave_n * NB + nb;
            return br < a.mblks && bc < cols ? (uint32_t)(br * all_cols + (pair ? nb * cols : 0) + bc) * 4096 + lane * 16 : share;
        };
        const __amdgpu_buffer_rsrc_t own = of(split);
#pragma unroll
        for (int mb = 0; mb < MB; mb++)
#pragma unroll
            for (int nb = 0; nb < NB; nb++)
#pragma unroll
                for (int r = 0; r < 16; r += 4)
                    put_partial(own, block_at(mb, nb) + r * 256, make_float4(out[mb][nb][r], out[mb][nb][r + 1], out[mb][nb][r + 2], out[mb][nb][r + 3]));
        if (!last_share(tickets + tm * a.seg[seg].strips + tn, shares, reinterpret_cast<uint32_t*>(sbuf))) return;
        // Shares 0 and 1 add in either order, so one of them stays where it is; a later one's sums are read back in their turn.  IN_FLIGHT
        // block rows of sums are requested at a time, of one share (one block row a wavefront: of as many shares).
        constexpr int IN_FLIGHT = MB == 4 ? 2 : 3;
        auto add = [&](int s, bool fresh, auto shares_tag) __attribute__((always_inline)) {
            constexpr int S = decltype(shares_tag)::value, ROWS = S > 1 ? 1 : MB < IN_FLIGHT ? MB : IN_FLIGHT;
#pragma unroll
            for (int mb0 = 0; mb0 < MB; mb0 += ROWS) {
                float4 v[S][ROWS][NB][4];
#pragma unroll
                for (int t = 0; t < S; t++)
#pragma unroll
                    for (int i = 0; i < ROWS; i++)
#pragma unroll
                        for (int nb = 0; nb < NB; nb++)
#pragma unroll
                            for (int r = 0; r < 4; r++) v[t][i][nb][r] = get_partial(of(s + t), block_at(mb0 + i, nb) + r * 1024);
#pragma unroll
                for (int t = 0; t < S; t++)
#pragma unroll
                    for (int i = 0; i < ROWS; i++)
#pragma unroll
                        for (int nb = 0; nb < NB; nb++)
#pragma unroll
                            for (int r = 0; r < 4; r++) {
                                const float4 f = v[t][i][nb][r];
                                f32x16_t& o = out[mb0 + i][nb];
                                o[4 * r] = fresh ? f.x : o[4 * r] + f.x;
                                o[4 * r + 1] = fresh ? f.y : o[4 * r + 1] + f.y;
                                o[4 * r + 2] = fresh ? f.z : o[4 * r + 2] + f.z;
                                o[4 * r + 3] = fresh ? f.w : o[4 * r + 3] + f.w;
                            }
            }
        };
        typedef std::integral_constant<int, 1> One;
        add(split == 0 ? 1 : 0, split > 1, One{});
        int s = split <= 1 ? 2 : 1;
        if constexpr (MB == 1)
#pragma nounroll
            for (; s + IN_FLIGHT <= shares; s += IN_FLIGHT) add(s, false, std::integral_constant<int, IN_FLIGHT>{});
#pragma nounroll
        for (; s < shares; s++) add(s, false, One{});
    }
    constexpr int CW = NB * 32;  // columns of the wavefront's tile
    static_assert(NWAVE * 32 * CW * 4 <= STAGES * A_STAGE + B_BUFS * B_STAGE, "staging area fits the stages");
    float* const stage = reinterpret_cast<float*>(lds) + wave * (32 * CW);
    const bool parts = partial && !tickets;  // partial tiles, for qmmh_reduce_kernel
    const int stride = parts && pair ? 2 * N : N;
    void* const ybase = parts ? static_cast<void*>(partial + (int64_t)split * a.M * stride) : a.seg[seg].y;
    const bool y_f32 = parts || a.out_f32 != 0;
    // COLS columns of the wavefront's tile leave together, eight consecutive ones per lane; `gated`: act(gate) * up of the two
    // column blocks.  (Partial tiles of a pair keep both sums: the gate columns of all outputs, then the up columns.)
    [[maybe_unused]] bool odd_one = false;  // this lane has stored a value that may not be finite
    auto store_tile = [&](auto gated_tag) {
        constexpr bool GATED = decltype(gated_tag)::value;
        constexpr int COLS = GATED ? CW / 2 : CW;
        constexpr int LPR = COLS / 8;     // lanes that share a row
        constexpr int RPP = kWave / LPR;  // rows per pass
        const int row_in = lane / LPR, c8 = (lane % LPR) * 8;
        const bool halves = pair && !GATED;
        const int n = n0 + (pair ? wave_n * 32 + (halves ? c8 % 32 : c8) : wave_n * CW + c8);
        const int col = halves && c8 >= 32 ? N + n : n;
        const bool wide = (reinterpret_cast<uintptr_t>(ybase) & 15) == 0 && (y_f32 ? (N & 3) == 0 : (N & 7) == 0);
#pragma unroll
        for (int mb = 0; mb < MB; mb++) {
            const int mtop = m0 + (wave_m * MB + mb) * 32;  // < mblks * 32 unless the whole block lies past the last row
#pragma unroll
            for (int r = 0; r < 16; r++) {
                const int at = (8 * (r >> 2) + 4 * h + (r & 3)) * COLS + j;
                if constexpr (GATED) {
                    stage[at] = fmul_unfused(act_value(a.act, out[mb][0][r]), out[mb][1][r]);
                } else {
#pragma unroll
                    for (int nb = 0; nb < NB; nb++) stage[at + nb * 32] = out[mb][nb][r];
                }
            }
#pragma unroll
            for (int p = 0; p < 32 / RPP; p++) {
                const int row = p * RPP + row_in;
                const int m = mtop + row;
                float4 lo = *reinterpret_cast<const float4*>(stage + row * COLS + c8);
                float4 hi = *reinterpret_cast<const float4*>(stage + row * COLS + c8 + 4);
                if (m >= mend || n >= N) continue;
                int64_t y_row = m;
                if (a.chunks) {
                    const int route = a.route_of[m];
                    if (route < 0) lo = hi = make_float4(0.f, 0.f, 0.f, 0.f);  // an expert id or a row of x out of range
                    y_row = route & INT32_MAX;
                }
                if (G32 && !parts)  // (one test for the eight; fix_output looks at each)
                    odd_one |= not_finite(((fabsf(lo.x) + fabsf(lo.y)) + (fabsf(lo.z) + fabsf(lo.w))) + ((fabsf(hi.x) + fabsf(hi.y)) + (fabsf(hi.z) + fabsf(hi.w))));
                const int64_t o = y_row * stride + col;
                if (wide && n + 8 <= N) {
                    if (y_f32) {
                        float4* dst = reinterpret_cast<float4*>(reinterpret_cast<float*>(ybase) + o);
                        dst[0] = lo;
                        dst[1] = hi;
                    } else {
                        uint4 u;
                        u.x = pack_bf16x2(lo.x, lo.y);
                        u.y = pack_bf16x2(lo.z, lo.w);
                        u.z = pack_bf16x2(hi.x, hi.y);
                        u.w = pack_bf16x2(hi.z, hi.w);
                        *reinterpret_cast<uint4*>(reinterpret_cast<uint16_t*>(ybase) + o) = u;
                    }
                } else {
                    const float v[8] = {lo.x, lo.y, lo.z, lo.w, hi.x, hi.y, hi.z, hi.w};
#pragma unroll
                    for (int e = 0; e < 8; e++) {
                        if (n + e < N) {
                            if (y_f32) {
                                reinterpret_cast<float*>(ybase)[o + e] = v[e];
                            } else {
                                reinterpret_cast<uint16_t*>(ybase)[o + e] = f32_to_bf16_bits(v[e]);
                            }
                        }
                    }
                }
            }
        }
    };
    if (pair && !parts) {
        store_tile(std::true_type{});
    } else {
        store_tile(std::false_type{});
    }
    if constexpr (G32) {
        // Dense groups of 32 keep what the any-width kernel makes of infinities: a lane goes over what it has stored once more.
        // (Partial tiles: qmmh_reduce_kernel does.)
        if (a.x && !parts && odd_one) {
            const int lanes = pair ? 4 : 8, row_in = lane / lanes, c8 = (lane % lanes) * 8;
            const int first = n0 + wave_n * (pair ? 32 : CW) + c8;
#pragma nounroll
            for (int r = row_in; r < MB * 32; r += kWave / lanes) {
                const int m = m0 + wave_m * MB * 32 + r;
#pragma nounroll
                for (int n = first; n < first + 8 && n < N && m < mend; n++) fix_output(a, a.seg[seg], m, n);
            }
        }
    }
}

// ---- adding the partial tiles of a K split --------------------------------------------------------------------------
// A matrix's partial tiles [ksplit][M][N] ([ksplit][M][gate N | up N] for a pair), added in split order; four columns a
// thread where N allows it.  grid.y: the matrices.
template <int V>
__global__ __launch_bounds__(256) void qmmh_reduce_kernel(const QmmHalfArgs a) {
    const QmmSegment& seg = a.seg[blockIdx.y];
    if (!seg.partial || seg.tickets) return;
    const int N = seg.N, stride = a.pair ? 2 * N : N, per_row = N / V;
    const int64_t total = (int64_t)a.M * per_row;
    const int64_t mn = (int64_t)a.M * stride;
    auto sum = [&](int64_t at, float (&v)[V]) {
        for (int s = 0; s < seg.ksplit; s++) {
            float t[V];
            if constexpr (V == 4) {
                const float4 f = *reinterpret_cast<const float4*>(seg.partial + (int64_t)s * mn + at);
                t[0] = f.x, t[1] = f.y, t[2] = f.z, t[3] = f.w;
            } else {
                t[0] = seg.partial[(int64_t)s * mn + at];
            }
#pragma unroll
            for (int i = 0; i < V; i++) v[i] = s ? v[i] + t[i] : t[i];
        }
    };
    for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < total; i += (int64_t)gridDim.x * 256) {
        const int m = (int)(i / per_row), c = (int)(i - (int64_t)m * per_row) * V;
        float v[V];
        sum((int64_t)m * stride + c, v);
        if (a.pair) {
            float u[V];
            sum((int64_t)m * stride + N + c, u);
#pragma unroll
            for (int e = 0; e < V; e++) v[e] = fmul_unfused(act_value(a.act, v[e]), u[e]);
        }
        const int64_t o = (int64_t)m * N + c;
        if (a.out_f32) {
#pragma unroll
            for (int e = 0; e < V; e++) static_cast<float*>(seg.y)[o + e] = v[e];
        } else {
#pragma unroll
            for (int e = 0; e < V; e++) static_cast<uint16_t*>(seg.y)[o + e] = f32_to_bf16_bits(v[e]);
        }
        float all = 0.0f;
#pragma unroll
        for (int e = 0; e < V; e++) all += fabsf(v[e]);
        if (a.x && not_finite(all)) {
#pragma nounroll
            for (int e = 0; e < V; e++) fix_output(a, seg, m, c + e);
        }
    }
}

// ---- variant table ----------------------------------------------------------------------------

typedef void (*QmmHalfKernel)(const QmmHalfArgs);
struct QmmHalfEntry {
    QmmVariant v;
    QmmHalfKernel fn, fn32;  // groups of 64 / 128, groups of 32
    int lds_bytes;
};

#define AQ_QMMH(PREFIX, BITS, MB, NB, WM, WN, ST, SE, SUFFIX)                                                        \
    {                                                                                                                            \
        {PREFIX #MB "_nb" #NB "_wm" #WM "_wn" #WN SUFFIX, BITS, MB, NB, WM, WN},                                                 \
            qmmh_kernel<BITS, MB, NB, WM, WN, ST, SE, 64>, qmmh_kernel<BITS, MB, NB, WM, WN, ST, SE, 32>, \
            ST*(WM * MB * 4096) + (BITS == 8 ? ST : 2) * (WN * NB * 32 * 64) + 2 * (WN * NB * 32) * SE * 2 +                      \
                (BITS == 4 && MB >= 3 ? WM * MB * 1024 : 0) + (half_rows_in_lds(BITS, MB, WM * WN) ? WM * MB * 128 : 0)          \
    }
#define AQ_QMMH4(...) AQ_QMMH("qmmh_b4_mb", 4, __VA_ARGS__)
#define AQ_QMMH8(...) AQ_QMMH("qmmh8_b8_mb", 8, __VA_ARGS__)

static const QmmHalfEntry kQmmHalfTable[] = {
    AQ_QMMH4(4, 2, 2, 2, 2, 16, "_s2c"),  // 256 x 128, four wavefronts, two stages (every LDS address a constant), one a CU
    AQ_QMMH4(4, 2, 1, 4, 2, 8, "_s2c"),  // 128 x 256, four wavefronts, two stages (every LDS address a constant), two a CU
    AQ_QMMH4(4, 2, 2, 4, 3, 16, ""),     // 256 x 256, eight wavefronts, three stages: an A tile feeds twice the MFMAs
    AQ_QMMH4(3, 2, 2, 4, 3, 16, ""),     // 192 x 256: a round of these takes 0.82 of a round of those; for row counts
                                                  // that fill their rounds better (1536 rows: 8 bands instead of 6 of 256)
    AQ_QMMH4(2, 2, 2, 2, 3, 16, ""),     // 128 x 128
    AQ_QMMH4(2, 2, 1, 4, 3, 16, ""),     // 64 x 256
    AQ_QMMH4(1, 2, 1, 4, 3, 8, ""),      // 32 x 256, three a CU
    // 8-bit codes (a wavefront's partial sums take 64 registers: 96 or 128 rows a wavefront would spill)
    AQ_QMMH8(2, 2, 2, 2, 3, 16, ""),      // 128 x 128
    AQ_QMMH8(2, 2, 2, 4, 3, 16, ""),     // 128 x 256, eight wavefronts
    AQ_QMMH8(2, 2, 1, 4, 3, 8, ""),
    AQ_QMMH8(1, 2, 1, 4, 3, 8, ""),
    AQ_QMMH8(1, 2, 2, 2, 3, 8, ""),      // 64 x 128 (4-bit tiles of that size, unsplit 167 -> 152 us on 509 x 15360 x 3840, lost to
                                                  // 128 x 128 and 192 x 256 with shares of K: 117 -> 142)
};

int qmmh_variant_count() { return (int)(sizeof(kQmmHalfTable) / sizeof(kQmmHalfTable[0])); }
const QmmVariant* qmmh_variant(int idx) {
    if (idx < 0 || idx >= qmmh_variant_count()) return nullptr;
    return &kQmmHalfTable[idx].v;
}
int qmmh_x_kind(int bits, int group_size) {
    return bits == 8 ? (group_size == 32 ? kXReadyHalf8G32 : kXReadyHalf8) : (group_size == 32 ? kXReadyHalf32 : kXReadyHalf);
}
int qmmh_rows(int idx) { return kQmmHalfTable[idx].v.wm * kQmmHalfTable[idx].v.mb * 32; }
// One share's partial sums of a matrix in 32 x 32 blocks, and a ticket for each of its tiles on the smallest kernels.
static size_t half_share_bytes(const QmmHalfCall& q, int i) {
    return (size_t)((q.M + 31) / 32) * ((q.seg[i].N + 31) / 32) * (q.pair ? 2 : 1) * 4096;
}
static size_t half_ticket_bytes(int M, int N) { return ((size_t)((M + 31) / 32) * ((N + 63) / 64) * 4 + 255) & ~(size_t)255; }
size_t qmmh_partial_bytes(const QmmHalfCall& q) {
    size_t bytes = 0;
    for (int i = 0; i < (q.pair ? 1 : q.nseg); i++)
        if (q.seg[i].ksplit > 1) bytes += half_share_bytes(q, i) * q.seg[i].ksplit + half_ticket_bytes(q.M, q.seg[i].N);
    return bytes;
}

// What a workgroup tile of each kernel takes: microseconds per 64-code block of K with one tile a CU on all CUs, the same per tile
// when CUs have more of them, outside the loop, and by how much of itself the loop is shorter when the rest of the chip idles (its
// clock and its share of L2).  First row: groups of 64 and 128, second: of 32.  Fitted to 2000 launches on weights from memory, 66 to
// 2048 rows (groups of 32: 509), K of 768 to 15360, 256 to 17664 columns, in 1 to 16 shares of K: predicted within 4 to 5 % (rms).
// What this picks takes 1 % longer than the best of a shape's measured forms; constants from K of 1024 and 4096, without groups of
// 32 and with shares at twice their cost took 2 to 4 %: 2048 x 14336 x 4096 unsplit 255 -> 234 in two shares, 509 x 15360 x 3840 in
// groups of 32 99 -> 94, 999 x 9920 x 4032 of 8 bit 159 -> 121.
struct QmmHalfCost {
    double solo, full, fixed, idle;
};
static const QmmHalfCost kQmmHalfCost[2][12] = {
    {{1.01, 1.13, 11.5, 0.21}, {1.00, 0.95, 12.0, 0.23}, {1.72, 1.98, 11.5, 0.38}, {1.23, 1.45, 12.5, 0.24}, {0.74, 0.59, 9.0, 0.26}, {0.78, 0.61, 9.5, 0.27},
     {0.55, 0.44, 8.5, 0.22}, {0.92, 0.65, 8.0, 0.21}, {1.22, 1.29, 9.5, 0.19}, {0.94, 0.69, 8.0, 0.23}, {0.73, 0.54, 7.0, 0.21}, {0.62, 0.43, 7.0, 0.20}},
    {{1.10, 1.19, 10.5, 0.13}, {1.16, 0.98, 11.5, 0.14}, {1.79, 1.92, 10.0, 0.24}, {1.29, 1.25, 11.0, 0.14}, {0.75, 0.62, 8.0, 0.18}, {0.87, 0.67, 8.5, 0.21},
     {0.65, 0.49, 7.5, 0.22}, {1.01, 0.71, 8.0, 0.14}, {1.38, 1.46, 10.0, 0.16}, {1.12, 0.80, 8.5, 0.16}, {0.89, 0.63, 7.0, 0.17}, {0.71, 0.50, 7.0, 0.18}}};
static_assert(sizeof(kQmmHalfCost[0]) / sizeof(kQmmHalfCost[0][0]) == sizeof(kQmmHalfTable) / sizeof(kQmmHalfTable[0]), "a cost for each kernel");

// Microseconds of kernel i over `tiles` tiles of `most` blocks at most and `all` blocks together.  (Matrices in one grid with different
// shares: at the most blocks for every tile, what this picked took 2 to 7 % longer than the best tile; here 0.2 to 1.5 %.)
static double half_cost(int i, int group_size, int64_t tiles, int most, int64_t all, int cus) {
    const QmmHalfCost& c = kQmmHalfCost[group_size == 32][i];
    const double load = (double)tiles / cus, per_cu = load > 1.0 ? ceil(load) : 1.0;
    const double longest = c.solo * most, full = per_cu > 1.0 ? c.full * per_cu * ((double)all / tiles) : 0.0;
    return c.fixed + (full > longest ? full : longest) * (1.0 - c.idle * (1.0 - load / per_cu));
}
static int64_t half_strips(int i, int N, bool pair) {
    const int bn = kQmmHalfTable[i].v.wn * kQmmHalfTable[i].v.nb * 32 / (pair ? 2 : 1);
    return (N + bn - 1) / bn;
}
static int64_t half_bands(int i, int M) { return (M + qmmh_rows(i) - 1) / qmmh_rows(i); }

void qmmh_split(int M, int K, int group_size, int bits, QmmSegment* seg, int cu_count) {
    const int cus = cu_count > 0 ? cu_count : 256;
    const int G = K / 64;
    // Matrices much wider than deep are one of a gated pair as often as not, whose grid has twice the tiles and partial tiles: theirs
    // cost the mean of the two.  150 pairs and as many single calls, against the single call's cost: pairs 1.1 % faster in the mean,
    // single calls 0.4 % slower; pairs of 71 x 2944 x 9984 42.3 -> 35.3 us, in groups of 32 of 8 bit 85 x 3328 x 7232 49.8 -> 42.3 and
    // 63 x 3840 x 15168 65.9 -> 59.3.  (At a pair's cost alone pairs are level with that and single calls another 1.5 % slower.)
    const bool paired = seg->N >= K + K / 2;
    double best_us = 1e30;
    seg->ksplit = 1;
    seg->gsplit = (G + 3) / 4 * 4;
    for (int i = 0; i < qmmh_variant_count(); i++) {
        if (kQmmHalfTable[i].v.bits != bits) continue;
        const int64_t tiles = half_bands(i, M) * half_strips(i, seg->N, false);
        for (int ks = 1; ks <= 16; ks++) {
            const int gsplit = ((G + ks - 1) / ks + 3) / 4 * 4;
            if (ks > 1 && (gsplit < 8 || tiles * ks > 4 * cus)) break;
            if (ks > 1 && (int64_t)(ks - 1) * gsplit >= G) continue;
            const int blocks = ks > 1 ? gsplit : G;
            double us = half_cost(i, group_size, tiles * ks, blocks, tiles * ks * blocks, cus);
            if (paired) {
                const int64_t both = half_bands(i, M) * half_strips(i, seg->N, true) * ks;
                us = 0.5 * (us + half_cost(i, group_size, both, blocks, both * blocks, cus));
            }
            // Partial tiles: one more launch, and their bytes (two of 2048 x 4096: 14 us for the sums, 10 for the stores).  Matrices of
            // few columns mostly stand in a grid beside wider ones, which fill the chip: there shares shorten little and cost the
            // same, so their bytes count for more (below 768 columns it is k and v rather than a layer's output).  Over 320 layers of
            // 66 to 2048 rows, against the bytes alone: q|k|v 1 to 2 % faster, o and down 0.1 % slower, the slowest layer against
            // q|k|v whole 5 -> 3 %; 1966 x 1920 x (2688, 576, 576) in groups of 32 64 -> 53 us, 1905 x 3648 x (1664, 704, 704) of
            // 8 bit 95 -> 80.  (1.6 up to 2048 columns: o and down 0.4 % slower again, 1053 x 2816 x 896 31 -> 37.)
            const double bytes_us = (double)ks * M * (double)seg->N * 4 / 2.4e6;
            if (ks > 1) us += 3.0 + bytes_us * (paired ? 1.5 : seg->N < 768 ? 1.6 : seg->N <= 2048 ? 1.3 : 1.0);
            if (us < best_us) best_us = us, seg->ksplit = ks, seg->gsplit = gsplit;
        }
    }
}

size_t qmmh_partial_most(int M, int K, int cu_count) {
    if (K / 64 <= 8) return 0;  // no share of fewer than eight blocks
    const int cus = cu_count > 0 ? cu_count : 256;
    // qmmh_split: strips x bands x shares <= 4 CUs, so that shares x N <= 4 CUs x columns of a tile / bands of M rows
    size_t most = 0;
    for (int i = 0; i < qmmh_variant_count(); i++) {
        const size_t rows = qmmh_rows(i), bn = (size_t)kQmmHalfTable[i].v.wn * kQmmHalfTable[i].v.nb * 32, blocks = ((size_t)M + 31) / 32 * 32;
        const size_t bytes = (size_t)4 * cus * bn * (blocks < rows ? blocks : rows) * 4 + half_ticket_bytes(M, (int)((size_t)4 * cus * bn / half_bands(i, M)) + 64);
        most = bytes > most ? bytes : most;
    }
    return (most + 255) & ~(size_t)255;
}

int qmmh_pick(const QmmHalfCall& q, int cu_count) {
    const int cus = cu_count > 0 ? cu_count : 256;
    int best = -1;
    double best_us = 1e30;
    for (int i = 0; i < qmmh_variant_count(); i++) {
        if (kQmmHalfTable[i].v.bits != q.bits) continue;
        int64_t tiles = 0, all = 0;
        int most = 0;
        for (int k = 0; k < (q.pair ? 1 : q.nseg); k++) {
            const int64_t t = half_bands(i, q.M) * half_strips(i, q.seg[k].N, q.pair) * q.seg[k].ksplit;
            const int b = q.seg[k].ksplit > 1 ? q.seg[k].gsplit : q.K / 64;
            tiles += t;
            all += t * b;
            most = b > most ? b : most;
        }
        double us = half_cost(i, q.group_size, tiles, most, all, cus);
        // Several 128 x 256 tiles of a pair a CU take 3 % longer than of one matrix (the costs come from single matrices; their epilogue has
        // no activation).  Over 70 pairs of 500 to 1600 rows: 1274 x 2048 x 7296 122 -> 117 us on 192 x 256, 1676 x 1536 x 5376
        // 99 -> 95, the largest loss against the costs before them 4 -> 2 %, the mean 0.1 % faster (at 5 and 7 % level).
        if (q.pair && kQmmHalfTable[i].v.mb == 4 && kQmmHalfTable[i].v.wm == 1 && tiles > cus) us *= 1.03;
        if (us < best_us) best_us = us, best = i;
    }
    return best;
}


// workspace: fragments, block sums, row factors (qmmt_workspace_bytes sizes them), then tickets and partial sums of shares of K
hipError_t qmmh_launch(int idx, const QmmHalfCall& q, void* workspace, hipStream_t stream) {
    if (idx < 0 || idx >= qmmh_variant_count() || q.nseg < 1 || q.nseg > kQmmSegments || (q.pair && q.nseg != 2)) return hipErrorInvalidValue;
    const QmmHalfEntry& e = kQmmHalfTable[idx];
    if (e.v.bits != q.bits) return hipErrorInvalidValue;
    const bool g32 = q.group_size == 32;
    const int rows = q.chunks ? q.most_rows : q.M;  // rows of the fragments
    const int mblks = (rows + 31) / 32;
    const size_t g4 = ((size_t)q.K / 64 + 3) / 4;
    uint16_t* xf = static_cast<uint16_t*>(workspace);
    uint16_t* xs = xf + (size_t)mblks * 32 * q.K;
    float* rs = reinterpret_cast<float*>(xs + (size_t)mblks * 32 * g4 * (g32 ? 16 : 8));
    hipError_t rc = hipSuccess;
    QmmHalfArgs a{};
    a.xf = xf;
    a.xs = xs;
    a.rs = rs;
    a.nseg = q.pair ? 1 : q.nseg;  // (a pair is one run of column units; the up matrix is a.seg[1])
    a.pair = q.pair;
    a.M = q.M;
    a.K = q.K;
    a.bits = q.bits;
    a.x = g32 && !q.chunks ? q.x : nullptr;
    a.gs_blocks = g32 ? 1 : q.group_size / 64;
    a.out_f32 = q.out_f32;
    a.act = q.act;
    a.mblks = mblks;
    const int bm = qmmh_rows(idx), bn = e.v.wn * e.v.nb * 32;
    char* const behind = static_cast<char*>(workspace) + ((qmmt_workspace_bytes(rows, q.K) + 255) & ~(size_t)255);
    uint32_t* const tickets = reinterpret_cast<uint32_t*>(behind);
    int count = 0;            // tickets
    size_t ticket_bytes = 0;  // that qmmh_partial_bytes has for them
    int split_segments = 0;   // whose partial tiles a second kernel adds
    int64_t split_work = 0;
    bool by4 = true;
    for (int i = 0; i < q.nseg; i++) {
        a.seg[i] = q.seg[i];
        if (a.seg[i].ksplit <= 1) a.seg[i].ksplit = 1, a.seg[i].gsplit = (q.K / 64 + 3) / 4 * 4;
    }
    if (!q.pair) std::stable_sort(a.seg, a.seg + q.nseg, [](const QmmSegment& l, const QmmSegment& r) { return l.gsplit > r.gsplit; });
    a.tiles_m = (rows + bm - 1) / bm;
    int64_t T = 0;  // tiles
    for (int i = 0; i < q.nseg; i++) {
        QmmSegment& seg = a.seg[i];
        seg.partial = nullptr;
        seg.tickets = nullptr;
        seg.strips = (int)half_strips(idx, seg.N, q.pair);
        if (q.pair && i == 1) break;
        T += (int64_t)(q.chunks ? q.most_chunks : a.tiles_m) * seg.strips * seg.ksplit;
        if (seg.ksplit > 1) {
            if (q.chunks || seg.gsplit % 4 != 0 || (int64_t)(seg.ksplit - 1) * seg.gsplit * 64 >= q.K) return hipErrorInvalidValue;
            ticket_bytes += half_ticket_bytes(q.M, seg.N);
            // Who adds the shares: the last workgroup of a tile where the others' sums are up to 100 KiB, else a kernel behind this one.  (A
            // CU reads some 18 KB a microsecond, the whole chip 4.5 TB/s behind a launch: 240 tiles of 128 x 128 in two shares 31.6 + 6.0
            // us -> 34.3, 116 of 192 x 256 82 + 10 -> 102.)  Over 40 layers of 66 to 2048 rows, against that kernel for all: limits of 48 / 64 / 100 /
            // 128 / 160 KiB 1.2 / 1.7 / 2.4 / 2.3 / 2.3 % faster, the slowest layer 1 / 1 / 0 / 1 / 5 % slower.
            if ((int64_t)(seg.ksplit - 1) * (bm < mblks * 32 ? bm : mblks * 32) * bn * 4 <= 100 << 10) {
                seg.tickets = tickets + count;
                count += a.tiles_m * seg.strips;
            } else {
                split_segments++;
                split_work = (int64_t)q.M * seg.N > split_work ? (int64_t)q.M * seg.N : split_work;
                by4 = by4 && seg.N % 4 == 0;
            }
        }
    }
    char* partial = behind + ticket_bytes;
    for (int i = 0; i < (q.pair ? 1 : q.nseg); i++) {
        QmmSegment& seg = a.seg[i];
        if (seg.ksplit <= 1) continue;
        seg.partial = reinterpret_cast<float*>(partial);
        partial += (size_t)mblks * ((seg.N + 31) / 32) * (q.pair ? 2 : 1) * 4096 * seg.ksplit;
    }
    if (q.x_ready != qmmh_x_kind(q.bits, q.group_size)) {
        typedef void (*PrepKernel)(const uint16_t*, uint16_t*, uint16_t*, float*, int, int, const int32_t*, const int32_t*, uint32_t*, int);
#define AQ_PREP(R) {{qmmh_prep_kernel<R, 64, 4>, qmmh_prep_kernel<R, 64, 8>}, {qmmh_prep_kernel<R, 32, 4>, qmmh_prep_kernel<R, 32, 8>}}
        static const PrepKernel kPrep[3][2][2] = {AQ_PREP(1), AQ_PREP(2), AQ_PREP(8)};
#undef AQ_PREP
        // rows a workgroup (us, 1 / 2 / 8): 256 x 4096 4.9 / 5.2 / 7.9, 256 x 15360 8.9 / 10.1 / 26; 509 x 4096 6.8 / 6.2 / 9.0, 1024 x
        // 15360 17.8 / 13.3 / 27; 2048 x 4096 14.7 / 11.9 / 9.9, 2048 x 15360 31.5 / 22.4 / 33
        const int log_rows = rows <= 256 ? 0 : rows >= 1536 && q.K <= 4096 ? 3 : 1;
        const PrepKernel fn = kPrep[log_rows == 3 ? 2 : log_rows][g32][q.bits == 8];
        hipLaunchKernelGGL(fn, dim3((unsigned)((mblks * 4 + 7) / 8 * 8 << (3 - log_rows))), dim3(kPrepThreads), 0, stream, q.x, xf, xs, rs, rows, q.K,
                           q.route_x, q.live_rows, tickets, count);
        rc = hipGetLastError();
        if (rc != hipSuccess) return rc;
    } else if (count > 0) {
        rc = fill_zero_launch(tickets, (size_t)count * 4, stream);
        if (rc != hipSuccess) return rc;
    }
    {
        // the patch an XCD's 32 CUs work on at a time: group_m row bands by the rest in column strips, fewest bytes per step
        // of K (4096 x 4096 x 16384: 598 -> 571 us against one band, 1024 x 4096 x 16384 on 64-row tiles 284 -> 201 us)
        const int at_once = 32 * (160 * 1024 / e.lds_bytes);
        int64_t least = INT64_MAX;
        a.group_m = 1;
        for (int gm = 1; gm <= a.tiles_m && gm <= at_once && !q.chunks; gm++) {
            const int64_t cost = (int64_t)gm * bm * 32 + (int64_t)((at_once + gm - 1) / gm) * bn * (2 * q.bits + 1);  // in 1/16 bytes: fp16 rows, 4.5- or 8.5-bit columns
            if (cost < least) least = cost, a.group_m = gm;
        }
    }
    a.chunks = q.chunks;
    a.nchunks = q.nchunks;
    a.route_of = q.route_of;
    a.expert_rows = q.expert_rows;
    a.row_base = q.row_base;
    a.row_base2 = q.row_base2;
    const unsigned grid = (unsigned)((T + 7) / 8 * 8);
    const QmmHalfKernel fn = g32 ? e.fn32 : e.fn;
    rc = ensure_dynamic_lds(reinterpret_cast<const void*>(fn), (size_t)e.lds_bytes);
    if (rc != hipSuccess) return rc;
    hipLaunchKernelGGL(fn, dim3(grid), dim3((unsigned)(e.v.wm * e.v.wn * kWave)), (size_t)e.lds_bytes, stream, a);
    rc = hipGetLastError();
    if (rc != hipSuccess || split_segments == 0) return rc;
    int64_t blocks = (split_work / (by4 ? 4 : 1) + 255) / 256;
    if (blocks > 4096) blocks = 4096;
    hipLaunchKernelGGL(by4 ? qmmh_reduce_kernel<4> : qmmh_reduce_kernel<1>, dim3((unsigned)blocks, (unsigned)a.nseg), dim3(256), 0, stream, a);
    return hipGetLastError();
}

}  // namespace aq
