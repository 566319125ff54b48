// Sums of shares of K inside the kernel that makes them: the workgroups of a tile store their partial sums, and the one that
// finishes last adds them up in the order of the shares and goes on to the epilogue.  No workgroup waits for another.  Against a
// kernel of its own behind the tiles that is one launch less, one share less to read back and, with several tiles a CU, the sums of
// some beside the products of others; but one CU reads all shares of a tile, which takes longer than the launch where they are large.
//
// The XCDs' L2 caches do not see each other's stores before the end of a kernel, so partial sums are stored and read with device
// scope, which goes past them, sixteen bytes a lane and 1 KiB a wavefront.  With all of them such, order is a matter of waits alone: a
// wavefront's stores have arrived where the others read (vmcnt) before the workgroup's barrier, and that lies before the ticket; the
// reads are issued behind the ticket's answer and a second barrier.  (A release and an acquire at the ticket also write back and drop
// the XCD's whole L2, weights that other workgroups are about to read included: a layer of 66 rows, 3072 / 8192, of 8 bit, 173 us so
// and 126 with waits, all shares added here.)
#ifndef AQ_SHARE_SUM_H
#define AQ_SHARE_SUM_H

#include "aq_device.h"

namespace aq {

// `bytes` of partial sums at `base` (below 4 GiB), four a lane; stores and reads past them are dropped and give zeros.
typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));
constexpr int kDeviceScope = 16;  // SC1
__device__ __forceinline__ __amdgpu_buffer_rsrc_t partial_sums(float* base, uint32_t bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(base, 0, bytes, 0x00020000);
}
__device__ __forceinline__ void put_partial(__amdgpu_buffer_rsrc_t to, uint32_t at, float4 v) {
    const u32x4_t u = {__float_as_uint(v.x), __float_as_uint(v.y), __float_as_uint(v.z), __float_as_uint(v.w)};
    __builtin_amdgcn_raw_buffer_store_b128(u, to, at, 0, kDeviceScope);
}
__device__ __forceinline__ float4 get_partial(__amdgpu_buffer_rsrc_t from, uint32_t at) {
    const u32x4_t u = __builtin_amdgcn_raw_buffer_load_b128(from, at, 0, kDeviceScope);
    return make_float4(__uint_as_float(u[0]), __uint_as_float(u[1]), __uint_as_float(u[2]), __uint_as_float(u[3]));
}

// True in every thread of the workgroup whose partial sums are the last of the tile's `shares` to be stored.  Called by all threads
// behind their stores; the ticket is zero before the kernel and again behind the last of them.  `flag`: a word of LDS that nothing
// else uses until the next barrier.
__device__ __forceinline__ bool last_share(uint32_t* ticket, int shares, uint32_t* flag) {
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // this wavefront's stores have arrived
    __syncthreads();
    if (threadIdx.x == 0) {
        const bool last = __hip_atomic_fetch_add(ticket, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == (uint32_t)shares - 1;
        if (last) __hip_atomic_store(ticket, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        *flag = last;
    }
    __syncthreads();
    return __builtin_amdgcn_readfirstlane(*flag) != 0;
}

}  // namespace aq

#endif
