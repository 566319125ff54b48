// What the kernels with fp16 operands (aq_qmm_half.hip, aq_qmm_routes.hip) share: rows of x and of the weights are brought into fp16's range
// by a power of two each, found from the largest magnitude of the row.
#ifndef AQ_FP16_OPERANDS_H
#define AQ_FP16_OPERANDS_H

#include "aq_device.h"

namespace aq {

// the value of lane `lane ^ BIT`
template <int BIT>
__device__ __forceinline__ float lane_xor(float v) {
    const int i = __float_as_int(v);
    if constexpr (BIT == 1) return __int_as_float(__builtin_amdgcn_mov_dpp(i, 0xb1, 0xf, 0xf, false));  // quad_perm 1 0 3 2
    if constexpr (BIT == 2) return __int_as_float(__builtin_amdgcn_mov_dpp(i, 0x4e, 0xf, 0xf, false));  // quad_perm 2 3 0 1
    if constexpr (BIT == 4) return __int_as_float(__builtin_amdgcn_ds_swizzle(i, 0x101f));
    if constexpr (BIT == 8) return __int_as_float(__builtin_amdgcn_mov_dpp(i, 0x128, 0xf, 0xf, false));  // row_ror 8
    if constexpr (BIT == 16) return __int_as_float(__builtin_amdgcn_permlane16_swap(i, i, false, false)[(threadIdx.x >> 4 & 1) ^ 1]);
    return __int_as_float(__builtin_amdgcn_permlane32_swap(i, i, false, false)[(threadIdx.x >> 5 & 1) ^ 1]);
}

// the largest value of the lanes that are BIT, 2 BIT, ... apart (by shuffles through LDS the pass over
// x of the matmul tiles made 29 layers of 66 to 414 rows 0.6 % slower)
template <int BIT>
__device__ __forceinline__ uint32_t max_lanes(uint32_t v) {
    if constexpr (BIT < kWave) {
        v = max(v, __float_as_uint(lane_xor<BIT>(__uint_as_float(v))));
        return max_lanes<2 * BIT>(v);
    }
    return v;
}

__device__ __forceinline__ uint32_t dup16(uint32_t h) { return (h & 0xffffu) | (h << 16); }

// 2^e for the largest finite magnitude `mag` (bf16 bits without the sign) such that mag * 2^e has binary
// exponent `target`; 1 for an all-zero row.  e is kept inside what fp32 powers of two hold.
__device__ __forceinline__ int exponent_shift(uint32_t mag, int target) {
    if (mag == 0) return 0;
    int e = target + 127 - (int)(mag >> 7);
    e = e > 120 ? 120 : e;
    e = e < -120 ? -120 : e;
    return e;
}
__device__ __forceinline__ float pow2f(int e) { return __uint_as_float((uint32_t)(127 + e) << 23); }

}  // namespace aq

#endif
