// MFMA matmul path (affine_qmm and the many-row calls of affine_qmv).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "aq_kernels.h"
#include "aq_workspace.h"

namespace aq {

// Largest M the dot2 matvec kernels take in one pass; a matmul call of up to this many rows runs as a matvec.
constexpr int kQmvMaxRows = 4;

struct QmmArgs {
    const uint16_t* x;  // [M, K] bf16
    const uint32_t* w;  // [N, K*bits/32]
    const uint16_t* s;  // [N, K/group]
    const uint16_t* b;  // [N, K/group]
    void* y;            // [M, N] bf16 or f32
    int M, K, N;
    int gs_blocks;  // 64-code blocks per quantisation group (1 for group 64, 2 for 128)
    int out_f32;
    const float* gate;  // not null: y = act(gate[m, n]) * (x . w^T)[m, n], gate being fp32 [M, N] (a gated MLP's other projection)
    int act;            // kActGeluTanh or kActSilu
    int x_ready;        // kXReady*: the workspace already holds this x as that pass over x leaves it (a call of several
                        // weight matrices against one x): the pass is skipped
};

// Which pass over x the workspace holds (QmmArgs.x_ready, and what a launch reports back through qmm_dispatch).
enum { kXReadyNone = 0, kXReadyTile4 = 1, kXReadyTile8 = 2, kXReadyHalf = 3, kXReadyHalf32 = 4, kXReadyHalf8 = 5, kXReadyHalf8G32 = 6 };

struct QmmVariant {
    const char* name;
    int bits;
    int mb, nb;  // 32x32 MFMA blocks per wavefront along M and N
    int wm, wn;  // wavefronts per workgroup along M and N
};

// Operands of the LDS-staged tile kernels (aq_qmm_tile.hip): x has been rewritten by their pass over x.
struct QmmTileArgs {
    const uint16_t* xf;  // activations in A-fragment order, rows padded to a multiple of 32
    const uint16_t* xs;  // per 64-code block sums of x as (hi, lo) bf16, four blocks per 16 bytes
    const float* rs;     // fp16-operand kernels: per row of x, the inverse of the power of two it was scaled by
    const uint32_t* w;
    const uint16_t* s;
    const uint16_t* b;
    void* y;
    int M, K, N;
    int gs_blocks;
    int out_f32;
    int mblks;             // ceil(M / 32)
    int tiles_m, tiles_n;  // workgroup tiles along M and N
    int ksplit;            // workgroups that share a tile along K (1: none)
    int gsplit;            // 64-code blocks of K per workgroup (a multiple of 4)
    float* partial;        // ksplit > 1: fp32 partial tiles [ksplit][M][N]
    const float* gate;     // as in QmmArgs (applied where the final value is stored)
    int act;
};

// (the variants of the fp16-operand kernels, aq_qmm_half.hip, are listed behind those of the tile kernels)
int qmmt_variant_count();
const QmmVariant* qmmt_variant(int idx);
// Device bytes the tile kernels need beside their operands for an M x K activation matrix.
size_t qmmt_workspace_bytes(int M, int K);
// Pass over x + tile kernel `idx`; `workspace` holds at least qmmt_workspace_bytes(M, K).
hipError_t qmmt_launch(int idx, const QmmArgs& a, void* workspace, hipStream_t stream);
// The pass over x variant idx needs (kXReady*).
int qmmt_x_kind(int idx);
int qmmt_half_index(int idx);  // the fp16-operand kernel (qmmh_variant) that a tile variant is, or -1
// The same with K shared out over ksplit workgroups per tile and a second kernel that adds the partial
// tiles: for few rows of x, where M x N tiles alone leave most of the chip idle.
size_t qmmt_splitk_bytes(int M, int N, int ksplit);
int qmmt_gsplit(int K, int ksplit);  // 64-code blocks of K per workgroup
hipError_t qmmt_launch_splitk(int idx, const QmmArgs& a, void* workspace, int ksplit, hipStream_t stream);

// Kernels for 5..64 rows of x whose LDS stages hold four blocks of K (aq_qmm_few.hip): listed behind the
// fp16-operand variants; they take the operands the tile kernels take and are launched through qmmt_launch_splitk.
int qmmf_variant_count();
const QmmVariant* qmmf_variant(int idx);
hipError_t qmmf_launch_kernel(int idx, const QmmTileArgs& a, hipStream_t stream);

// Kernels with fp16 matrix-core operands (aq_qmm_half.hip): 4 bit, scale * (code - 8); 8 bit, code - 128.  Same workspace.
constexpr int kQmmSegments = 8;  // weight matrices of one call
struct QmmSegment {
    const uint32_t* w;
    const uint16_t* s;
    const uint16_t* b;
    void* y;
    int N;
    int ksplit, gsplit;    // workgroups that share a tile along K, 64-code blocks of K each takes (qmmh_split)
    int strips;            // filled by the launcher: column strips
    float* partial;        // filled by the launcher: partial sums of shares of K, or null
    uint32_t* tickets;     // one for each tile
};
struct QmmHalfArgs {
    const uint16_t* xf;  // as in QmmTileArgs, fp16
    const uint16_t* xs;
    const float* rs;  // per row, the inverse of the power of two it was scaled by
    const uint16_t* x;  // groups of 32 (not expert slabs): x itself, for outputs without a finite value; else null
    QmmSegment seg[kQmmSegments];
    int nseg, pair;  // pair: seg[0] is the gate matrix, seg[1] the up matrix of a gated MLP; one output
    int M, K;
    int bits, gs_blocks, out_f32, act;
    int mblks, tiles_m;
    int group_m;  // row bands of a group of tiles
    // routes grouped by expert (aq_moe_group.hip), or null
    const RouteChunk* chunks;
    const int32_t* nchunks;
    const int32_t* route_of;
    int expert_rows, row_base, row_base2;
};
struct QmmHalfCall {
    const uint16_t* x;
    int M, K, group_size, bits;
    QmmSegment seg[kQmmSegments];
    int nseg, pair, act, out_f32;
    int x_ready;  // kXReady*
    const RouteChunk* chunks;  // expert slabs: most_chunks and most_rows bound what the lists on the device hold
    const int32_t *nchunks, *route_x, *route_of, *live_rows;
    int most_chunks, most_rows, expert_rows, row_base, row_base2;
};
// The tile that workgroup `place` of a grid works on: the matrix (negative: none), the tile's number in it, the matrix's column units
// (strips x shares of K: each share stores fp32 partial tiles).  Workgroups are dealt to the 8 XCDs round-robin, so every 8th one
// shares an L2.  Each XCD has a contiguous run of the tiles of every matrix; what is left over of a matrix goes to the XCDs behind
// those that the one before it ended with.  (One run over the tiles of all matrices gave q's long ones to the first XCDs and the short
// shares of k and v to the others.  us with the sums of shares, that -> this, 8 bit on 64 x 128 tiles: 777 x 2560 x (2048, 512, 512),
// k and v in five shares, 58 -> 38; 562 x 2816 x (2496, 1152, 1152) in six 93 -> 46.)
struct QmmTileAt {
    int seg, id, units;
};
__host__ __device__ inline QmmTileAt qmmh_tile_at(const QmmSegment* seg, int nseg, int row_bands, int place) {
    int in_run = place >> 3, ends = 0;
    for (int i = 0; i < nseg; i++) {
        const int units = seg[i].strips * seg[i].ksplit, tiles = row_bands * units, left = tiles & 7;
        const int xcd = (place - ends) & 7, run = (tiles >> 3) + (xcd < left);
        if (in_run < run) return {i, xcd * (tiles >> 3) + (xcd < left ? xcd : left) + in_run, units};
        in_run -= run;
        ends += left;
    }
    return {-1, 0, 0};
}
int qmmh_variant_count();
const QmmVariant* qmmh_variant(int idx);
int qmmh_x_kind(int bits, int group_size);  // the pass over x their kernels need (kXReady*)
int qmmh_rows(int idx);  // rows of x of a workgroup tile
hipError_t qmmh_launch(int idx, const QmmHalfCall& q, void* workspace, hipStream_t stream);
// How a matrix of seg->N columns shares K out for M rows of x: a function of M, K, N, the group size and the code width alone, so that
// the call of several matrices, the gated pair and a call of its own add in the same order and give the same bytes.
void qmmh_split(int M, int K, int group_size, int bits, QmmSegment* seg, int cu_count);
// The kernel for these matrices (the bytes of a result do not depend on it).
int qmmh_pick(const QmmHalfCall& q, int cu_count);
size_t qmmh_partial_bytes(const QmmHalfCall& q);
// What one matrix of any N needs at most with up to M rows of up to K columns.
size_t qmmh_partial_most(int M, int K, int cu_count);

// Routes grouped by expert on tiles of up to 48 routes in blocks of 16 (aq_qmm_routes.hip), 4-bit codes.
constexpr int kRouteRows = 48;  // routes of a chunk
struct QmmRouteArgs {
    const uint16_t* xf;  // [rows][K up to a multiple of 256] fp16
    const uint32_t* xs;  // [rows][groups up to a multiple of 16] sums of x, two bf16 each
    const float* rs;     // [rows] the inverse of the power of two a row was scaled by
    const uint32_t* w;
    const uint16_t *s, *b;
    void* y;
    int K, N, pair, act, out_f32;
    int by_route;  // rows of xf are the routes (else the rows of x)
    int strips, most_chunks, expert_rows, row_base, row_base2;
    const RouteChunk* chunks;
    const int32_t *route_x, *route_of;
};
struct QmmRouteCall {
    const uint16_t* x;
    int rows, by_route;  // of the copy of x
    const uint32_t* w;
    const uint16_t *s, *b;
    void* y;
    int K, N, group_size, pair, act, out_f32, expert_rows, row_base, row_base2;
    RouteGroupArgs lists;  // chunks of kRouteRows, runs side by side
};
// Whether the tiles of such a call take a matrix (rows: of the copy of x), and what they keep in scratch.
int qmmr_strips(int N, bool pair);  // workgroups an expert's chunk of routes takes
bool qmmr_fits(int rows, int K, int N, int group_size, int bits);
size_t qmmr_workspace_bytes(int rows, int K, int group_size);
// Lists, pass over x and tiles.
hipError_t qmmr_launch(const QmmRouteCall& c, void* workspace, hipStream_t stream);

hipError_t fill_zero_launch(void* p, size_t bytes, hipStream_t stream);

// Upper bound (256-byte aligned) of the workspace bytes qmm_dispatch may use for an M x K by N call: the
// rewritten activations and, for few rows, the fp32 partial tiles of the K split.  Callers that keep their
// own data in the same workspace place it behind this.
size_t qmm_scratch_bytes(int M, int K, int N, int cu_count);

// Sizes ws for prefill calls with activations of up to M x K ahead of time (not during capture).
int qmm_reserve(hipStream_t stream, Workspace* ws, int M, int K, int cu_count, FailFn fail);

// Validated-shape dispatch used by aq_qmm and by aq_qmv for calls the matvec families pass on.
// Returns an AQ_* / hipError_t code through `fail`.
// `forced` indexes the tile variants (qmmt_variant), or is negative.
// gate (fp32 [M, N], or null) and act: the gated-MLP epilogue, see QmmArgs; only where qmm_takes_gate says so.
// x_state (or null): in, which pass over this x the workspace already holds (kXReady*); out, which it holds now.
int qmm_dispatch(hipStream_t stream, Workspace* ws, int cu_count, int forced, const char** last_variant, const void* x,
                 const void* packed, const void* scales, const void* biases, void* y, int M, int K, int N,
                 int group_size, int bits, bool out_f32, FailFn fail, const float* gate = nullptr, int act = 0,
                 int* x_state = nullptr);
// Whether the fp16-operand kernels take a call (4- or 8-bit codes, groups of 32, 64 or 128, K a multiple of 64).
bool qmmh_takes(const void* x, const void* packed, int K, int group_size, int bits);
// Whether an unforced call on one matrix runs on them (the choice among the families by shape).
bool qmmh_runs(int M, int K, int N, int group_size, int bits);
// One call of them over q.nseg matrices, or on expert slabs (idx < 0: qmmh_pick); x_state as in qmm_dispatch.  Scratch that
// cannot be had (the stream is being captured, or there is no memory): kQmmhNoScratch, nothing launched.
constexpr int kQmmhNoScratch = INT32_MIN;
int qmmh_run(hipStream_t stream, Workspace* ws, int cu_count, int idx, QmmHalfCall& q, const char** last_variant, FailFn fail, int* x_state);
// Whether qmm_dispatch runs this call on the tile kernels, whose stores can carry the gated-MLP epilogue.
bool qmm_takes_gate(const void* x, const void* packed, int K, int group_size, int bits);

}  // namespace aq
