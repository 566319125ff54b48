// The token-tile kernels of aq_qmv_tok.h for 4-bit codes, the sum of partial tiles, and the host side of both widths: choice and
// launch.
#include "aq_qmv_tok.h"

#include <cmath>

namespace aq {

static const QmvTokEntry kEntries4[kTokPerWidth] = {AQ_QMVT_SET(4, 2)};
const QmvTokEntry* tok_entries_4() { return kEntries4; }

static const QmvTokEntry& tok_entry(int idx) { return idx < kTokPerWidth ? tok_entries_4()[idx] : tok_entries_8()[idx - kTokPerWidth]; }

int qmvt_variant_count() { return 2 * kTokPerWidth; }
const QmvVariant* qmvt_variant(int idx) {
    if (idx < 0 || idx >= qmvt_variant_count()) return nullptr;
    return &tok_entry(idx).v;
}

static bool tok_whole_runs(const QmvArgs& a) { return a.gs_shift == 6 && a.K % 256 == 0; }
static int tok_runs_of(const TokArgs& a) { return a.ksplit > 1 ? a.share : (a.K + 255) / 256; }
// LDS of a workgroup whose longest share is `runs` runs.  The wavefronts' sums meet behind what is staged (red_at) where that costs no
// workgroup of a CU, else in its place, behind a barrier (us, in its place / behind: 4 / 16 / 32 rows of 4096 x 14336, 8 bit 14.6 /
// 16.3 / 20.2 against 14.4 / 16.1 / 19.9, 4 bit 16 / 32 rows 11.6 / 16.3 against 11.5 / 16.1).
// (inside: the sums of shares that a workgroup works through by itself lie behind, for the scales are needed again)
static size_t tok_lds_bytes(const QmvTokEntry& e, bool g32, int runs, uint32_t* red_at = nullptr, bool inside = false) {
    const size_t staged = tok_sb_bytes(g32, e.wg_rows, runs) + (size_t)kTokWaves * tok_own_bytes(e.v.bits, g32, e.ts);
    const size_t sums = (size_t)kTokWaves * 16 * e.ts * e.wg_rows * 4, cu = 160 * 1024;
    const int of_a_cu = e.v.rows * e.ts <= 2 ? 2 : 1;  // workgroups that a CU's registers hold
    if (inside) {
        if (red_at) *red_at = (uint32_t)staged;
        return staged + sums + sums / kTokWaves;
    }
    const bool behind = staged + sums <= cu / of_a_cu;
    if (red_at) *red_at = behind ? (uint32_t)staged : 0;
    return behind ? staged + sums : staged > sums ? staged : sums;
}

bool qmvt_fits(const TokArgs& a, int bits, int group_size, int idx, bool exact_only) {
    const QmvVariant* v = qmvt_variant(idx);
    if (!v || bits != v->bits || (group_size != 32 && group_size != 64 && group_size != 128)) return false;
    // (K up to 16384: what the tests cover; longer rows go to the kernels that split K)
    if (a.M < 1 || (a.M > v->m && (exact_only || a.M > kTokMax || a.tokens < 1 || a.tokens > v->m)) || a.N < 1 || a.K < 64 || a.K % 64 != 0 || a.K > kTokMaxK) return false;
    const uintptr_t al16 = reinterpret_cast<uintptr_t>(a.x) | reinterpret_cast<uintptr_t>(a.w) | reinterpret_cast<uintptr_t>(a.w2);
    if (al16 & 15) return false;
    // 32-bit byte offsets into the packed matrix and into x
    if ((uint64_t)a.N * (uint64_t)(a.K * bits / 8) >= (1ull << 32)) return false;
    // (scales of any alignment would do; which calls run here by it is kept: 8 bytes where K is whole runs in groups of 64, else 16)
    const uintptr_t sb = reinterpret_cast<uintptr_t>(a.s) | reinterpret_cast<uintptr_t>(a.b) | reinterpret_cast<uintptr_t>(a.s2) |
                         reinterpret_cast<uintptr_t>(a.b2);
    const bool exact = tok_whole_runs(a) && (sb & 7) == 0;
    if (!exact && (exact_only || (sb & 15))) return false;
    return tok_lds_bytes(tok_entry(idx), group_size == 32, tok_runs_of(a), nullptr, a.inside > 1) <= 160 * 1024;
}

const char* qmvt_name(int idx, const TokArgs& a) { return tok_entry(idx).name[a.gs_shift == 5 ? 2 : tok_whole_runs(a) ? 0 : 1]; }

static int tok_blocks(const QmvTokEntry& e, int M, int tokens, int N, bool pair, int ksplit) {
    const int outs = e.wg_rows / (pair ? 2 : 1);
    const int blocks = (N + outs - 1) / outs * (ksplit > 1 ? ksplit : 1), parts = (M + tokens - 1) / tokens;
    return parts > 1 ? (blocks + 7) / 8 * 8 * parts : blocks;
}
int qmvt_tokens(int M) { return M <= 32 ? M : (M + 1) / 2; }

static hipError_t tok_reduce_one(const TokArgs& a, int bits, bool pair, hipStream_t stream) {
    if (a.ksplit <= 1) return hipSuccess;
    TokReduceArgs r{};
    r.x = a.x;
    r.M = a.M;
    r.K = a.K;
    r.bits = bits;
    r.gs_shift = a.gs_shift;
    r.out_f32 = a.out_f32;
    r.act = a.act;
    r.pair = pair;
    r.count = 1;
    r.w[0] = a.w, r.s[0] = a.s, r.b[0] = a.b;
    r.w[1] = a.w2, r.s[1] = a.s2, r.b[1] = a.b2;
    r.y[0] = a.y;
    r.N[0] = a.N;
    r.ksplit[0] = a.ksplit;
    r.tile[0] = a.tile;
    return tok_reduce_launch(r, stream);
}

static hipError_t tok_launch(int idx, TokArgs a, bool pair, hipStream_t stream) {
    const QmvTokEntry& e = tok_entry(idx);
    if (a.tokens < 1) a.tokens = a.M;
    const bool g32 = a.gs_shift == 5;
    const QmvTokKernel fn = pair ? e.pair[g32] : e.fn[g32];
    const size_t lds = tok_lds_bytes(e, g32, tok_runs_of(a), &a.red_at);
    if (hipError_t rc = ensure_dynamic_lds(reinterpret_cast<const void*>(fn), lds)) return rc;
    hipLaunchKernelGGL(fn, dim3((unsigned)tok_blocks(e, a.M, a.tokens, a.N, pair, a.ksplit)), dim3((unsigned)(e.v.waves * kWave)), lds, stream, a);
    if (hipError_t rc = hipGetLastError()) return rc;
    return tok_reduce_one(a, e.v.bits, pair, stream);
}

hipError_t qmvt_launch(int idx, const TokArgs& a, hipStream_t stream) {
    if (idx < 0 || idx >= qmvt_variant_count()) return hipErrorInvalidValue;
    return tok_launch(idx, a, false, stream);
}

hipError_t qmvt_multi_launch(int idx, TokMultiArgs ma, int bits, hipStream_t stream) {
    if (idx < 0 || idx >= qmvt_variant_count() || ma.count < 1 || ma.count > kQmvMultiMax) return hipErrorInvalidValue;
    const QmvTokEntry& e = tok_entry(idx);
    const bool g32 = ma.common.gs_shift == 5;
    const QmvTokMultiKernel fn = e.multi[g32];
    int blocks = 0, runs = 1;
    TokReduceArgs r{};
    r.x = ma.common.x;
    r.M = ma.common.M;
    r.K = ma.common.K;
    r.bits = bits;
    r.gs_shift = ma.common.gs_shift;
    r.out_f32 = ma.common.out_f32;
    r.count = ma.count;
    bool split = false, inside = false;
    for (int i = 0; i < ma.count; i++) {
        blocks += tok_blocks(e, ma.common.M, ma.tokens, ma.N[i], false, ma.ksplit[i]);
        ma.block_end[i] = blocks;
        const int n = ma.ksplit[i] > 1 ? ma.share[i] : (ma.common.K + 255) / 256;
        runs = n > runs ? n : runs;
        split |= ma.ksplit[i] > 1;
        inside |= ma.inside[i] > 1;
        r.w[i] = ma.w[i], r.s[i] = ma.s[i], r.b[i] = ma.b[i];
        r.y[i] = ma.y[i];
        r.N[i] = ma.N[i];
        r.ksplit[i] = ma.ksplit[i];
        r.tile[i] = ma.ksplit[i] > 1 ? ma.tile[i] : nullptr;
    }
    const size_t lds = tok_lds_bytes(e, g32, runs, &ma.red_at, inside);
    if (lds > 160 * 1024 || (inside && e.v.rows > kTokInsideSets)) return hipErrorInvalidValue;
    if (hipError_t rc = ensure_dynamic_lds(reinterpret_cast<const void*>(fn), lds)) return rc;
    hipLaunchKernelGGL(fn, dim3((unsigned)blocks), dim3((unsigned)(e.v.waves * kWave)), lds, stream, ma);
    if (hipError_t rc = hipGetLastError()) return rc;
    return split ? tok_reduce_launch(r, stream) : hipSuccess;
}

bool qmvt_pair_supported(int idx) { return idx >= 0 && idx < qmvt_variant_count() && tok_entry(idx).pair[0] != nullptr; }

hipError_t qmvt_pair_launch(int idx, const TokArgs& a, hipStream_t stream) {
    if (!qmvt_pair_supported(idx)) return hipErrorInvalidValue;
    return tok_launch(idx, a, true, stream);
}

bool qmvt_grouped_fits(const QmvArgs& a, int bits, int group_size, bool pair) {
    if ((bits != 4 && bits != 8) || (group_size != 32 && group_size != 64 && group_size != 128)) return false;
    if (a.N < 1 || a.K < 64 || a.K % 64 != 0 || a.K % group_size != 0 || a.K > kTokMaxK) return false;
    const uintptr_t al = reinterpret_cast<uintptr_t>(a.x) | reinterpret_cast<uintptr_t>(a.w) | reinterpret_cast<uintptr_t>(a.s) |
                         reinterpret_cast<uintptr_t>(a.b);
    if (al & 15) return false;
    // 32-bit byte offsets into an expert's rows and into x
    if ((uint64_t)a.expert_rows * (uint64_t)(a.K * bits / 8) >= (1ull << 32) || (uint64_t)a.x_rows * (uint64_t)a.K * 2 >= (1ull << 32)) return false;
    // (which slabs run here is kept: those whose first row's scales lie on 16 bytes)
    const int64_t groups = a.K / group_size;
    if ((a.expert_rows * groups) % 8 || (a.row_base * groups) % 8 || (pair && (a.row_base2 * groups) % 8)) return false;
    return tok_lds_bytes(tok_entry(1), group_size == 32, (a.K + 255) / 256) <= 160 * 1024;
}

hipError_t qmvt_grouped_launch(int bits, int tokens, bool pair, int most_chunks, TokArgs a, hipStream_t stream) {
    const int idx = (bits == 8 ? kTokPerWidth : 0) + (tokens == 32 ? 5 : 1);  // (four sets of rows: the second of a token count)
    const QmvTokEntry& e = tok_entry(idx);
    const bool g32 = a.gs_shift == 5;
    const QmvTokKernel fn = e.grouped[g32][pair ? 1 : 0];
    if (!fn || e.v.m != tokens) return hipErrorInvalidValue;
    const size_t lds = tok_lds_bytes(e, g32, (a.K + 255) / 256, &a.red_at);
    if (hipError_t rc = ensure_dynamic_lds(reinterpret_cast<const void*>(fn), lds)) return rc;
    const int outs = e.wg_rows / (pair ? 2 : 1);
    hipLaunchKernelGGL(fn, dim3((unsigned)((a.N + outs - 1) / outs), (unsigned)most_chunks), dim3((unsigned)(e.v.waves * kWave)), lds, stream, a);
    return hipGetLastError();
}

size_t qmvt_tile_bytes(int M, int N, bool pair, int ksplit) {
    return ksplit > 1 ? ((size_t)ksplit * M * N * (pair ? 2 : 1) * 4 + 255) & ~(size_t)255 : 0;
}

// Microseconds of a call: `fixed` (launch, first requests, the meeting in LDS and the store), and per pass of a workgroup (eight
// runs of 256 codes) `pass` for x and `set` for each of its sets of 16 weight rows.  From runs at K = 2048 to 12288 with one to eight
// sets in 208 workgroups, 12 and 24 rows of x (graph replay over 640 MB of weights; off by 2.5 to 5.5 % rms, 14 % at most).
struct TokCost {
    double fixed, pass, set;
};
constexpr double kMeetFixed = 0.4, kMeetSet = 0.15;  // a meeting in LDS between shares that a workgroup works through by itself
static const TokCost& tok_cost(int bits, int group_size, int tokens) {
    // [8 bit][groups of 32][more than 16 rows of x]
    static const TokCost kCost[2][2][2] = {{{{2.6, 1.25, 0.72}, {2.8, 2.5, 0.89}}, {{3.0, 1.13, 0.93}, {3.85, 2.1, 1.43}}},
                                           {{{2.3, 1.34, 1.27}, {2.45, 2.6, 1.37}}, {{2.6, 1.4, 1.35}, {2.9, 2.8, 1.5}}}};
    return kCost[bits == 8][group_size == 32][tokens > 16];
}
// Passes of a workgroup whose share is `runs` runs (a part of a pass costs more than its part).
static double tok_passes(int runs) {
    return runs > kTokWaves ? 0.5 * ((runs + kTokWaves - 1) / kTokWaves + (double)runs / kTokWaves) : 1.0;
}
static double tok_time(const TokCost& c, int rs, const TokPart& p, int K) {
    if (p.inside <= 1) return tok_passes(p.runs) * (c.pass + rs * c.set);
    const int last = (K + 255) / 256 - (p.inside - 1) * p.runs;
    return ((p.inside - 1) * tok_passes(p.runs) + tok_passes(last)) * (c.pass + rs * c.set) + (p.inside - 1) * (kMeetFixed + kMeetSet * rs);
}
// When the last CU is done with these matrices on `rs` sets a workgroup, one workgroup a CU at a time, in the order of the grid.
static double tok_span(const TokCost& c, int rs, const TokPart* parts, int count, int K, int parts_of_x, int cus) {
    struct Level {  // CUs that are free at a time, earliest first
        double at;
        int64_t cus;
    };
    if (count == 1)
        return (double)(((parts[0].sets + rs - 1) / rs * parts[0].shares * parts_of_x + cus - 1) / cus) * tok_time(c, rs, parts[0], K);
    // Halves of the rows of x: the two workgroups of a band are on one XCD, and every member begins at the first, which therefore has
    // the most of them (64 rows of 9600 x (5248 | 1344 | 1344): 248 workgroups, but 34 of them on the 32 CUs there, 74 us for 37)
    const int xcds = parts_of_x > 1 ? 8 : 1;
    cus = cus > xcds ? cus / xcds : 1;
    Level levels[4 * kQmvMultiMax] = {{0.0, cus}};
    int n = 1;
    for (int i = 0; i < count; i++) {
        const double t = tok_time(c, rs, parts[i], K);
        int64_t groups = ((parts[i].sets + rs - 1) / rs * parts[i].shares + xcds - 1) / xcds * parts_of_x;
        while (groups > 0) {
            if (n == 1) {  // whole rounds
                levels[0].at += (double)(groups / cus) * t;
                groups %= cus;
                if (groups == 0) break;
            }
            const int64_t now = groups < levels[0].cus ? groups : levels[0].cus;
            const Level next = {levels[0].at + t, now};
            if ((levels[0].cus -= now) == 0) {
                n--;
                for (int l = 0; l < n; l++) levels[l] = levels[l + 1];
            }
            int at = 0;
            while (at < n && levels[at].at < next.at) at++;
            if (at < n && levels[at].at == next.at) {
                levels[at].cus += now;
            } else if (n == 4 * kQmvMultiMax) {  // (not seen: as if they were done when those above are)
                levels[at < n ? at : n - 1].cus += now;
            } else {
                for (int l = n++; l > at; l--) levels[l] = levels[l - 1];
                levels[at] = next;
            }
            groups -= now;
        }
    }
    return levels[n - 1].at;
}
// Sets of 16 weight rows per workgroup, by the same figures.  Mostly the fewest that leave every CU one workgroup (us on one, two,
// four, eight sets; 24 rows of x, K = 2816, groups of 64: 4096 rows of weights 8.3 / 9.6 / 11.9 / 17.2, 8192 15.1 / 10.0 / 12.1 /
// 17.2, 14336 27.9 / 18.1 / 12.3 / 17.4, 2 x 14336 35.1 / 23.9 / 18.3 from two on); fewer where a second round would be nearly empty,
// and where members of a grid differ in length, so that the ones that are not shared out do not outlast the rest.
// (a pair has two or more, one of each matrix)
static int tok_sets(const TokCost& c, const TokPart* parts, int count, int K, int parts_of_x, bool pair, int cus, double* us = nullptr) {
    double best = 1e30;
    int best_rs = 1, most = 8;
    for (int i = 0; i < count; i++)
        if (parts[i].inside > 1) most = kTokInsideSets;
    for (int rs = pair ? 2 : 1; rs <= most; rs *= 2) {
        const double t = tok_span(c, rs, parts, count, K, parts_of_x, cus);
        if (t < best) best = t, best_rs = rs;
    }
    if (us) *us = c.fixed + best;
    return best_rs;
}

// Shares of K where a workgroup would make three passes or more: the shares' workgroups carry more rows each, and a second launch
// adds their partial tiles, which costs about 2.5 us and one more per megabyte (us, whole / shares, 12 and 24 rows of x: 4096 x 14336
// 16.3 / 13.3 and 26.6 / 17.8, 1024 x 14336 16.3 / 8.6 and 26.6 / 10.7, 1536 x 6144 8.5 / 8.4 and 13.0 / 10.4).  With two passes they
// win at more than 16 rows what they lose at fewer, and lose where a matrix is one of several in a grid (1024 x 4096 6.5 / 7.2 and
// 9.6 / 8.6; 32 rows of 4096 x (4096 | 1024 | 1024) 13.2 / 16.3).
// The choice for every call of up to 32 rows is the one that 12 and 24 rows are fastest with together, and the one for 48 rows beyond,
// so that shares, and with them the bytes of a row, do not depend on the number of rows.
void qmvt_split(int bits, int group_size, int M, int K, int N, bool pair, int cu_count, int* ksplit, int* share) {
    const int cus = cu_count > 0 ? cu_count : 256, quads = (K + 255) / 256, most = M <= 32 ? 32 : 64;
    *ksplit = 1;
    *share = quads;
    if ((bits != 4 && bits != 8) || M > kTokMax || K % 64 != 0 || K > kTokMaxK) return;  // (no call of these kernels)
    if (quads <= 2 * kTokWaves) return;
    double best = 1e30;
    for (int ks = 1; ks <= kTokShares && ks <= quads; ks++) {
        const int sh = (quads + ks - 1) / ks, n = (quads + sh - 1) / sh;
        if (n != ks || qmvt_tile_bytes(most, N, pair, n) > kTokTileBytes) continue;
        double sum = 0.0;
        for (const int rows : {12, 24, 48}) {
            if ((rows > 32) != (M > 32)) continue;
            const int tokens = qmvt_tokens(rows);
            const TokPart part{(int64_t)((N + 15) / 16) * (pair ? 2 : 1), n, sh, 0};
            double us;
            tok_sets(tok_cost(bits, group_size, tokens), &part, 1, K, (rows + tokens - 1) / tokens, pair, cus, &us);
            // (a tenth: no shares for next to nothing, see above; not from 33 rows on, where 44 shapes that it decides take 5 % more
            // with it: 64 rows of 8 bit by 16320 x 8061 67.0 / 81.2 us, but 48 by 12416 x 5650 in groups of 32 54.3 / 47.2)
            if (n > 1) us = (M <= 32 ? 1.1 : 1.0) * us + 2.5 + (double)qmvt_tile_bytes(rows, N, pair, n) / 1e6;
            sum += us;
        }
        if (sum < best) best = sum, *ksplit = n, *share = sh;
        if (sh <= kTokWaves) break;  // (one pass: more shares have nothing to win)
    }
}

int qmvt_pick(int bits, int group_size, int M, int K, const TokPart* parts, int count, bool pair, int cu_count, double* us) {
    if (M < 1 || M > kTokMax || K < 64 || K % 64 != 0 || K > kTokMaxK || count < 1) return -1;
    const int cus = cu_count > 0 ? cu_count : 256, tokens = qmvt_tokens(M), most = tokens <= 16 ? 16 : 32;
    int rs = tok_sets(tok_cost(bits, group_size, tokens), parts, count, K, (M + tokens - 1) / tokens, pair, cus, us), runs = 1;
    bool inside = false;
    for (int i = 0; i < count; i++) {
        const int n = parts[i].inside > 1 ? (K + 255) / 256 : parts[i].runs;
        runs = n > runs ? n : runs;
        inside |= parts[i].inside > 1;
    }
    for (int i = 0; i < qmvt_variant_count(); i++) {  // (listed with eight, four, two, one sets)
        const QmvTokEntry& e = tok_entry(i);
        if (e.v.bits != bits || e.v.m != most || e.v.rows > rs) continue;
        if (tok_lds_bytes(e, group_size == 32, runs, nullptr, inside) <= 160 * 1024) return i;
    }
    return -1;
}

// V columns a thread.  grid.y: the matrices.
template <int V>
__global__ __launch_bounds__(256) void tok_reduce_kernel(const TokReduceArgs a) {
    const int mi = blockIdx.y;
    const float* const tile = a.tile[mi];
    if (!tile) return;
    const int N = a.N[mi], shares = a.ksplit[mi], stride = a.pair ? 2 * N : N;
    const int64_t mn = (int64_t)a.M * stride;
    const int per_row = N / V;
    auto sum = [&](int64_t at, float (&v)[V]) {
        float t[kTokShares][V];
#pragma unroll
        for (int s = 0; s < kTokShares; s++) {  // (requested together: a chain of loads is a chain of latencies)
            if (s >= shares) break;
            if constexpr (V == 4) {
                const float4 f = *reinterpret_cast<const float4*>(tile + s * mn + at);
                t[s][0] = f.x, t[s][1] = f.y, t[s][2] = f.z, t[s][3] = f.w;
            } else {
                t[s][0] = tile[s * mn + at];
            }
        }
#pragma unroll
        for (int s = 0; s < kTokShares; s++)
            if (s < shares)
#pragma unroll
                for (int e = 0; e < V; e++) v[e] = s ? v[e] + t[s][e] : t[s][e];
    };
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= (int64_t)a.M * per_row) return;
    const int m = (int)(i / per_row), c = (int)(i - (int64_t)m * per_row) * V;
    float v[V], u[V];
    sum((int64_t)m * stride + c, v);
    if (a.pair) sum((int64_t)m * stride + N + c, u);
#pragma unroll
    for (int e = 0; e < V; e++) {
        if (a.gs_shift == 5) {  // (dense groups of 32 keep what the any-width kernel makes of infinities)
#pragma nounroll
            for (int part = 0; part < (a.pair ? 2 : 1); part++) {
                if (!not_finite(part ? u[e] : v[e])) continue;
                const int mat = a.pair ? part : mi;
                const size_t row = (size_t)(c + e), groups = (size_t)(a.K >> 5);
                const float f = plain_dot_g32(a.x + (size_t)m * a.K, a.w[mat] + row * (size_t)(a.K / 32 * a.bits), a.s[mat] + row * groups,
                                              a.b[mat] + row * groups, a.K, a.bits);
                if (part) u[e] = f; else v[e] = f;
            }
        }
        if (a.pair) v[e] = fmul_unfused(act_value(a.act, v[e]), u[e]);
        const int64_t at = (int64_t)m * N + c + e;
        if (a.out_f32)
            static_cast<float*>(a.y[mi])[at] = v[e];
        else
            static_cast<uint16_t*>(a.y[mi])[at] = f32_to_bf16_bits(v[e]);
    }
}

hipError_t tok_reduce_launch(const TokReduceArgs& a, hipStream_t stream) {
    int64_t most = 0;
    // (groups of 32: outputs that are formed again take a thread each, on as many CUs as there are wavefronts; us, by fours in
    // workgroups of 256 / so: 4 rows with an infinity by 2684 x 10112 3810 / 734, 25 by 625 x 15616 1790 / 1281)
    bool by4 = a.gs_shift != 5;
    for (int i = 0; i < a.count; i++) {
        if (!a.tile[i]) continue;
        most = (int64_t)a.M * a.N[i] > most ? (int64_t)a.M * a.N[i] : most;
        by4 = by4 && a.N[i] % 4 == 0;
    }
    if (most == 0) return hipSuccess;
    const int threads = a.gs_shift == 5 ? 64 : 256;
    const int64_t grid = (most / (by4 ? 4 : 1) + threads - 1) / threads;
    hipLaunchKernelGGL(by4 ? tok_reduce_kernel<4> : tok_reduce_kernel<1>, dim3((unsigned)grid, (unsigned)a.count), dim3((unsigned)threads), 0, stream, a);
    return hipGetLastError();
}

}  // namespace aq
