// The two device steps on either side of the expert-gathered projections.
//
// moe_route_kernel: per token row, the top-k experts by (score descending, expert id ascending), their
//   softmax weights and the route -> token map, written as the int32 / float32 arrays aq_gather_qmv reads.
//   Selection and weights follow rocm_moe_router (go/engine/hip/kernels/moe/routing.hipinc:3-77) and the
//   host router it shadows, hipGemma4MoEBatchRouteGroups (go/engine/hip/hip_gemma4_moe.go:294-366):
//   softmax over the selected scores, times an optional per-expert scale.  With normalise off the weights
//   are the softmax over ALL experts gathered at the selection (hipQwen3MoERouterSelect,
//   go/engine/hip/hip_qwen3_moe_router.go:25-88).  The reference copies the scores to the host, groups
//   routes by expert and uploads chunks every step; here nothing leaves the device.
//
// moe_combine_kernel: out[row, :] = sum over ranks of route_rows[row*top_k + rank, :] * weight, ranks
//   ascending, the product rounded to fp32 before it is added: rocm_moe_batch_scatter_routes followed by
//   rocm_moe_batch_reduce_routes (routing.hipinc:100-158).  With bf16 steps every product and every partial
//   sum is rounded to bf16, the chain lthn_moe_weighted_sum_bf16 reproduces
//   (go/engine/metal/kernels/moe/lthn_moe_weighted_sum.metal:17-38).
//
// One wavefront per token row; expert scores sit in registers, lane l holding experts l, l+64, ...
#include <cfloat>
#include <climits>

#include "aq_device.h"
#include "aq_kernels.h"

namespace aq {

// Wave-wide maximum / minimum through DPP inside each row of 16 lanes (old value = the identity for lanes a
// pattern leaves without a source) and SGPR reads across the four rows.
__device__ __forceinline__ float wave_max_f32(float v) {
    const int ninf = __float_as_int(-INFINITY);
    v = fmaxf(v, __int_as_float(__builtin_amdgcn_update_dpp(ninf, __float_as_int(v), 0xB1, 0xF, 0xF, false)));
    v = fmaxf(v, __int_as_float(__builtin_amdgcn_update_dpp(ninf, __float_as_int(v), 0x4E, 0xF, 0xF, false)));
    v = fmaxf(v, __int_as_float(__builtin_amdgcn_update_dpp(ninf, __float_as_int(v), 0x141, 0xF, 0xF, false)));
    v = fmaxf(v, __int_as_float(__builtin_amdgcn_update_dpp(ninf, __float_as_int(v), 0x140, 0xF, 0xF, false)));
    const float a = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), 0));
    const float b = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), 16));
    const float c = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), 32));
    const float d = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), 48));
    return fmaxf(fmaxf(a, b), fmaxf(c, d));
}
__device__ __forceinline__ int wave_min_i32(int v) {
    v = min(v, __builtin_amdgcn_update_dpp(INT_MAX, v, 0xB1, 0xF, 0xF, false));
    v = min(v, __builtin_amdgcn_update_dpp(INT_MAX, v, 0x4E, 0xF, 0xF, false));
    v = min(v, __builtin_amdgcn_update_dpp(INT_MAX, v, 0x141, 0xF, 0xF, false));
    v = min(v, __builtin_amdgcn_update_dpp(INT_MAX, v, 0x140, 0xF, 0xF, false));
    return min(min(__builtin_amdgcn_readlane(v, 0), __builtin_amdgcn_readlane(v, 16)),
               min(__builtin_amdgcn_readlane(v, 32), __builtin_amdgcn_readlane(v, 48)));
}

template <int PER>
__global__ __launch_bounds__(256) void moe_route_kernel(const MoeRouteArgs a) {
    const int lane = threadIdx.x & (kWave - 1);
    const int row = blockIdx.x * 4 + (threadIdx.x >> 6);
    if (row >= a.rows) return;  // whole wavefronts leave together
    const int E = a.num_experts;

    float v[PER];
    bool open[PER];  // in range and not yet selected
#pragma unroll
    for (int j = 0; j < PER; j++) {
        const int e = lane + j * kWave;
        open[j] = e < E;
        float s = -INFINITY;
        if (open[j]) {
            s = a.logits_bf16 ? bf16_bits_to_f32(static_cast<const uint16_t*>(a.logits)[(int64_t)row * E + e])
                              : static_cast<const float*>(a.logits)[(int64_t)row * E + e];
            if (s != s) s = -INFINITY;  // a NaN score never wins a comparison; rank it last
        }
        v[j] = s;
    }

    float all_max = 0.0f, all_total = 1.0f;
    if (!a.normalise) {
        float m = -INFINITY;
#pragma unroll
        for (int j = 0; j < PER; j++)
            if (open[j]) m = fmaxf(m, v[j]);
        all_max = wave_max_f32(m);
        float t = 0.0f;
#pragma unroll
        for (int j = 0; j < PER; j++)
            if (open[j]) t += expf(v[j] - all_max);
        all_total = wave_sum(t);
        if (all_total == 0.0f) all_total = 1.0f;
    }

    int my_id = 0;
    float my_score = 0.0f;
    for (int k = 0; k < a.top_k; k++) {
        float bv = -INFINITY;
        int bi = INT_MAX;
#pragma unroll
        for (int j = 0; j < PER; j++) {
            // ascending expert id inside a lane, so the strict comparison keeps the lowest id of equals
            if (open[j] && (bi == INT_MAX || v[j] > bv)) {
                bv = v[j];
                bi = lane + j * kWave;
            }
        }
        const float best = wave_max_f32(bv);
        const int winner = wave_min_i32((bi != INT_MAX && bv == best) ? bi : INT_MAX);
        if ((winner & (kWave - 1)) == lane) {
#pragma unroll
            for (int j = 0; j < PER; j++)
                if (j == (winner >> 6)) open[j] = false;
        }
        if (lane == k) {
            my_id = winner;
            my_score = best;
        }
    }

    const bool mine = lane < a.top_k;
    float p;
    if (a.normalise) {
        // the first selection holds the largest score
        const float top = __shfl(my_score, 0, kWave);
        const float e = mine ? expf(my_score - top) : 0.0f;
        const float sum = wave_sum(e);
        p = sum > 0.0f ? e / sum : 0.0f;
    } else {
        p = expf(my_score - all_max) / all_total;
    }
    if (mine) {
        if (a.expert_scales) p *= a.expert_scales[my_id];
        const int64_t o = (int64_t)row * a.top_k + lane;
        a.ids[o] = my_id;
        a.weights[o] = p;
        if (a.token_of_route) a.token_of_route[o] = row;
    }
}

__global__ __launch_bounds__(256) void moe_combine_kernel(const MoeCombineArgs a) {
#pragma clang fp contract(off)  // the product is rounded before it is added, as the two reference kernels do
    const int64_t total = (int64_t)a.rows * a.n;
    for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < total; i += (int64_t)gridDim.x * 256) {
        const int row = (int)(i / a.n);
        const int col = (int)(i - (int64_t)row * a.n);
        float acc = 0.0f;
#pragma unroll 8
        for (int r = 0; r < a.top_k; r++) {
            const int64_t pair = (int64_t)row * a.top_k + r;
            const float y = a.in_f32 ? static_cast<const float*>(a.route_rows)[pair * a.n + col]
                                     : bf16_bits_to_f32(static_cast<const uint16_t*>(a.route_rows)[pair * a.n + col]);
            float w = a.weights[pair];
            if (a.bf16_steps) {
                w = bf16_bits_to_f32(f32_to_bf16_bits(w));
                const float scaled = bf16_bits_to_f32(f32_to_bf16_bits(y * w));
                acc = r == 0 ? scaled : bf16_bits_to_f32(f32_to_bf16_bits(acc + scaled));
            } else {
                const float scaled = y * w;
                acc = acc + scaled;
            }
        }
        if (a.out_f32) {
            static_cast<float*>(a.out)[i] = acc;
        } else {
            static_cast<uint16_t*>(a.out)[i] = f32_to_bf16_bits(acc);
        }
    }
}

// The same for bf16 route rows of whole 16-byte pieces: one row per grid row, eight columns a thread, AHEAD ranks at a time.
// Bound: latency; rows and weights of the AHEAD ranks are requested together, ahead of any use and with no branch between them
// (ranks past the last repeat it and are not added).
// Roundings by instruction and chosen at compile time: with f32_to_bf16_bits and its NaN case inside, and a break after the last
// rank, the weights were loaded rank by rank between thousands of branches (us a pass: 8 tokens, 8 of 128 experts, 2816 columns
// 79.6 -> 77.8, 512 tokens 243.8 -> 241.0; one element a thread: 18 for the kernel alone at 512 tokens).
// As many ranks at a time as there are, up to eight: repeated ones cost their loads.
template <int AHEAD, bool STEPS>
__global__ __launch_bounds__(kWave) void moe_combine_wide_kernel(const MoeCombineArgs a) {
#pragma clang fp contract(off)  // as above
    const int col = ((int)blockIdx.x * kWave + (int)threadIdx.x) * 8;
    if (col >= a.n) return;
    const int64_t row = blockIdx.y, first = row * a.top_k;
    const uint16_t* const src = static_cast<const uint16_t*>(a.route_rows) + first * a.n + col;
    float acc[8] = {0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f};
    auto rounded = [](float (&v)[2]) {
        const uint32_t u = pack_bf16x2(v[0], v[1]);
        v[0] = __uint_as_float(u << 16), v[1] = __uint_as_float(u & 0xffff0000u);
    };
    for (int r0 = 0; r0 < a.top_k; r0 += AHEAD) {
        uint4 v[AHEAD];
        float w[AHEAD];
#pragma unroll
        for (int i = 0; i < AHEAD; i++) {
            const int r = min(r0 + i, a.top_k - 1);
            v[i] = *reinterpret_cast<const uint4*>(src + (int64_t)r * a.n);
            w[i] = a.weights[first + r];
        }
#pragma unroll
        for (int i = 0; i < AHEAD; i++) {
            const bool counts = r0 + i < a.top_k;  // (a break here, and every load moves down to its use)
            float wi = w[i];
            if (STEPS) wi = bf16_bits_to_f32(f32_to_bf16_bits(wi));
            const uint32_t words[4] = {v[i].x, v[i].y, v[i].z, v[i].w};
#pragma unroll
            for (int c = 0; c < 4; c++) {
                float term[2] = {__uint_as_float(words[c] << 16) * wi, __uint_as_float(words[c] & 0xffff0000u) * wi};
                if (STEPS) rounded(term);
                float sum[2] = {acc[2 * c] + term[0], acc[2 * c + 1] + term[1]};
                if (STEPS) {
                    rounded(sum);
                    if (r0 + i == 0) sum[0] = term[0], sum[1] = term[1];  // (not 0 + term: minus zero stays)
                }
                acc[2 * c] = counts ? sum[0] : acc[2 * c], acc[2 * c + 1] = counts ? sum[1] : acc[2 * c + 1];
            }
        }
    }
    if (a.out_f32) {
        float4* const dst = reinterpret_cast<float4*>(static_cast<float*>(a.out) + row * a.n + col);
        dst[0] = make_float4(acc[0], acc[1], acc[2], acc[3]);
        dst[1] = make_float4(acc[4], acc[5], acc[6], acc[7]);
    } else {
        *reinterpret_cast<uint4*>(static_cast<uint16_t*>(a.out) + row * a.n + col) =
            make_uint4(pack_bf16x2(acc[0], acc[1]), pack_bf16x2(acc[2], acc[3]), pack_bf16x2(acc[4], acc[5]), pack_bf16x2(acc[6], acc[7]));
    }
}

hipError_t moe_route_launch(const MoeRouteArgs& a, hipStream_t stream) {
    if (a.rows <= 0) return hipSuccess;
    if (a.num_experts <= 0 || a.num_experts > kMoeMaxExperts || a.top_k <= 0 || a.top_k > kMoeMaxTopK ||
        a.top_k > a.num_experts)
        return hipErrorInvalidValue;
    const dim3 grid((unsigned)((a.rows + 3) / 4)), block(256);
    const int per = (a.num_experts + kWave - 1) / kWave;
    if (per <= 1) {
        hipLaunchKernelGGL(moe_route_kernel<1>, grid, block, 0, stream, a);
    } else if (per <= 2) {
        hipLaunchKernelGGL(moe_route_kernel<2>, grid, block, 0, stream, a);
    } else if (per <= 4) {
        hipLaunchKernelGGL(moe_route_kernel<4>, grid, block, 0, stream, a);
    } else if (per <= 8) {
        hipLaunchKernelGGL(moe_route_kernel<8>, grid, block, 0, stream, a);
    } else {
        hipLaunchKernelGGL(moe_route_kernel<16>, grid, block, 0, stream, a);
    }
    return hipGetLastError();
}

hipError_t moe_combine_launch(const MoeCombineArgs& a, hipStream_t stream) {
    const int64_t total = (int64_t)a.rows * a.n;
    if (total <= 0) return hipSuccess;
    const uintptr_t at = reinterpret_cast<uintptr_t>(a.route_rows) | reinterpret_cast<uintptr_t>(a.out);
    if (!a.in_f32 && a.n % 8 == 0 && (at & 15) == 0 && a.rows <= 65535) {
        typedef void (*CombineKernel)(MoeCombineArgs);
        static const CombineKernel kWide[3][2] = {{moe_combine_wide_kernel<2, false>, moe_combine_wide_kernel<2, true>},
                                                  {moe_combine_wide_kernel<4, false>, moe_combine_wide_kernel<4, true>},
                                                  {moe_combine_wide_kernel<8, false>, moe_combine_wide_kernel<8, true>}};
        const CombineKernel fn = kWide[a.top_k <= 2 ? 0 : a.top_k <= 4 ? 1 : 2][a.bf16_steps ? 1 : 0];
        hipLaunchKernelGGL(fn, dim3((unsigned)((a.n / 8 + kWave - 1) / kWave), (unsigned)a.rows), dim3(kWave), 0, stream, a);
        return hipGetLastError();
    }
    int64_t blocks = (total + 255) / 256;
    if (blocks > 8192) blocks = 8192;
    hipLaunchKernelGGL(moe_combine_kernel, dim3((unsigned)blocks), dim3(256), 0, stream, a);
    return hipGetLastError();
}

}  // namespace aq
