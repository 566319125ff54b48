// The token-tile kernels of aq_qmv_tok.h for 4-bit codes, and the host side of both widths: choice and launch.
#include "aq_qmv_tok.h"

namespace aq {

static const QmvTokEntry kEntries4[kTokPerWidth] = {AQ_QMVT_SET(4)};
const QmvTokEntry* tok_entries_4() { return kEntries4; }

static const QmvTokEntry& tok_entry(int idx) { return idx < kTokPerWidth ? tok_entries_4()[idx] : tok_entries_8()[idx - kTokPerWidth]; }

int qmvt_variant_count() { return 2 * kTokPerWidth; }
const QmvVariant* qmvt_variant(int idx) {
    if (idx < 0 || idx >= qmvt_variant_count()) return nullptr;
    return &tok_entry(idx).v;
}

// (of a gated pair: one form for both matrices, so the alignment of either decides it)
static int tok_form(const QmvArgs& a) {
    const uintptr_t al8 = reinterpret_cast<uintptr_t>(a.s) | reinterpret_cast<uintptr_t>(a.b) | reinterpret_cast<uintptr_t>(a.s2) |
                          reinterpret_cast<uintptr_t>(a.b2);
    if (a.gs_shift == 6 && a.K % 256 == 0 && (al8 & 7) == 0) return kTokExact;
    return a.gs_shift == 5 ? kTokG32 : kTokAny;
}
static size_t tok_lds_bytes(const QmvTokEntry& e, int K, int form) {
    const size_t scales = (size_t)e.wg_rows * ((K + 255) / 256 + 1) * (form == kTokG32 ? 32 : 16);
    if (form == kTokExact) return scales + (size_t)e.lds;
    return scales > (size_t)e.lds ? scales : (size_t)e.lds;
}

bool qmvt_fits(const QmvArgs& a, int bits, int group_size, int idx, bool exact_only) {
    const QmvVariant* v = qmvt_variant(idx);
    if (!v || bits != v->bits || (group_size != 32 && group_size != 64 && group_size != 128)) return false;
    // (K up to 16384, as qmvt_pick has it: what the tests cover; longer rows go to the kernels that split K)
    if (a.M < 1 || a.M > v->m || a.N < 1 || a.K < 64 || a.K % 64 != 0 || a.K > kTokMaxK) return false;
    const uintptr_t al16 = reinterpret_cast<uintptr_t>(a.x) | reinterpret_cast<uintptr_t>(a.w) | reinterpret_cast<uintptr_t>(a.w2);
    if (al16 & 15) return false;
    // 32-bit byte offsets into the packed matrix and into x
    if ((uint64_t)a.N * (uint64_t)(a.K * bits / 8) >= (1ull << 32)) return false;
    const QmvTokEntry& e = tok_entry(idx);
    const int form = tok_form(a);
    if (form == kTokExact) {
        if (e.wg_rows * (a.K / 256) > tok16_stage_pieces(v->waves) * v->waves * kWave) return false;
    } else {
        const uintptr_t sb = reinterpret_cast<uintptr_t>(a.s) | reinterpret_cast<uintptr_t>(a.b) | reinterpret_cast<uintptr_t>(a.s2) |
                             reinterpret_cast<uintptr_t>(a.b2);
        if (exact_only || (sb & 15)) return false;
    }
    return tok_lds_bytes(e, a.K, form) <= 160 * 1024;
}

const char* qmvt_name(int idx, const QmvArgs& a) { return tok_entry(idx).name[tok_form(a)]; }

hipError_t qmvt_launch(int idx, const QmvArgs& a, hipStream_t stream) {
    if (idx < 0 || idx >= qmvt_variant_count()) return hipErrorInvalidValue;
    const QmvTokEntry& e = tok_entry(idx);
    const int form = tok_form(a);
    const QmvTokKernel fn = e.fn[form];
    const size_t lds = tok_lds_bytes(e, a.K, form);
    if (hipError_t rc = ensure_dynamic_lds(reinterpret_cast<const void*>(fn), lds)) return rc;
    const int wg_rows = e.wg_rows;
    hipLaunchKernelGGL(fn, dim3((unsigned)((a.N + wg_rows - 1) / wg_rows)), dim3((unsigned)(e.v.waves * kWave)), lds, stream, a);
    return hipGetLastError();
}

hipError_t qmvt_multi_launch(int idx, QmvMultiArgs ma, hipStream_t stream) {
    if (idx < 0 || idx >= qmvt_variant_count() || ma.count < 1 || ma.count > kQmvMultiMax) return hipErrorInvalidValue;
    const QmvTokEntry& e = tok_entry(idx);
    int form = kTokExact;
    for (int i = 0; i < ma.count; i++) {
        QmvArgs one = ma.common;
        one.s = ma.s[i];
        one.b = ma.b[i];
        const int f = tok_form(one);
        form = f > form ? f : form;
    }
    const QmvTokMultiKernel fn = e.multi[form];
    const size_t lds = tok_lds_bytes(e, ma.common.K, form);
    if (hipError_t rc = ensure_dynamic_lds(reinterpret_cast<const void*>(fn), lds)) return rc;
    int blocks = 0;
    for (int i = 0; i < ma.count; i++) {
        blocks += (ma.N[i] + e.wg_rows - 1) / e.wg_rows;
        ma.block_end[i] = blocks;
    }
    hipLaunchKernelGGL(fn, dim3((unsigned)blocks), dim3((unsigned)(e.v.waves * kWave)), lds, stream, ma);
    return hipGetLastError();
}

bool qmvt_pair_supported(int idx) { return idx >= 0 && idx < qmvt_variant_count() && tok_entry(idx).pair[0] != nullptr; }

hipError_t qmvt_pair_launch(int idx, const QmvArgs& a, hipStream_t stream) {
    if (!qmvt_pair_supported(idx)) return hipErrorInvalidValue;
    const QmvTokEntry& e = tok_entry(idx);
    const int form = tok_form(a);
    const QmvTokKernel fn = e.pair[form];
    const size_t lds = tok_lds_bytes(e, a.K, form);
    if (hipError_t rc = ensure_dynamic_lds(reinterpret_cast<const void*>(fn), lds)) return rc;
    const int outs = e.wg_rows / 2;
    hipLaunchKernelGGL(fn, dim3((unsigned)((a.N + outs - 1) / outs)), dim3((unsigned)(e.v.waves * kWave)), lds, stream, a);
    return hipGetLastError();
}

bool qmvt_grouped_fits(const QmvArgs& a, int bits, int group_size, bool pair) {
    if ((bits != 4 && bits != 8) || (group_size != 32 && group_size != 64 && group_size != 128)) return false;
    if (a.N < 1 || a.K < 64 || a.K % 64 != 0 || a.K % group_size != 0 || a.K > kTokMaxK) return false;
    const uintptr_t al = reinterpret_cast<uintptr_t>(a.x) | reinterpret_cast<uintptr_t>(a.w) | reinterpret_cast<uintptr_t>(a.s) |
                         reinterpret_cast<uintptr_t>(a.b);
    if (al & 15) return false;
    // 32-bit byte offsets into an expert's rows and into x
    if ((uint64_t)a.expert_rows * (uint64_t)(a.K * bits / 8) >= (1ull << 32) || (uint64_t)a.x_rows * (uint64_t)a.K * 2 >= (1ull << 32)) return false;
    // an expert's scales are read in 16-byte pieces from its first row on
    const int64_t groups = a.K / group_size;
    if ((a.expert_rows * groups) % 8 || (a.row_base * groups) % 8 || (pair && (a.row_base2 * groups) % 8)) return false;
    return tok_lds_bytes(tok_entry(0), a.K, group_size == 32 ? kTokG32 : kTokAny) <= 160 * 1024;
}

hipError_t qmvt_grouped_launch(int bits, int tokens, bool pair, int most_chunks, const QmvArgs& a, hipStream_t stream) {
    const int idx = (bits == 8 ? kTokPerWidth : 0) + (tokens == 32 ? 3 : 0);  // (four sets of rows: the first of a token count)
    const QmvTokEntry& e = tok_entry(idx);
    const int form = a.gs_shift == 5 ? kTokG32 : kTokAny;
    const QmvTokKernel fn = e.grouped[form == kTokG32][pair ? 1 : 0];
    if (!fn || e.v.m != tokens) return hipErrorInvalidValue;
    const size_t lds = tok_lds_bytes(e, a.K, form);
    if (hipError_t rc = ensure_dynamic_lds(reinterpret_cast<const void*>(fn), lds)) return rc;
    const int outs = e.wg_rows / (pair ? 2 : 1);
    hipLaunchKernelGGL(fn, dim3((unsigned)((a.N + outs - 1) / outs), (unsigned)most_chunks), dim3((unsigned)(e.v.waves * kWave)), lds, stream, a);
    return hipGetLastError();
}

// The variant for `rows` weight rows in all, or -1.
int qmvt_pick(int bits, int M, int K, int rows, int cu_count) {
    if (M < 1 || M > kTokMax || K < 64 || K % 64 != 0 || K > kTokMaxK) return -1;
    const int cus = cu_count > 0 ? cu_count : 256;
    // eight wavefronts, one run each per pass; one set of 16 tokens up to 16 rows of x, else two; as many sets of 16
    // weight rows per workgroup (fewer reads of x) as still leave three quarters of the CUs a workgroup
    const int most = M <= 16 ? 16 : 32;
    const int rs = (rows + 63) / 64 >= (cus * 3) / 4 ? 4 : (rows + 31) / 32 >= (cus * 3) / 4 ? 2 : 1;
    for (int i = 0; i < qmvt_variant_count(); i++) {
        const QmvVariant& v = tok_entry(i).v;
        if (v.bits == bits && v.m == most && v.rows == rs) return i;
    }
    return -1;
}
// The same for the gated pair of two matrices of N rows each (at least two sets of rows: one of either).
int qmvt_pick_pair(int bits, int M, int K, int N, int cu_count) {
    const int idx = qmvt_pick(bits, M, K, 2 * N, cu_count);
    if (idx < 0 || qmvt_pair_supported(idx)) return idx;
    return idx - 1;  // (the entries of a token count are listed with 4, 2, 1 sets)
}

}  // namespace aq
