// Raw buffer accesses of the sweeps (device).
#pragma once

#include <hip/hip_runtime.h>
#include <cstdint>

namespace m4g {

// Raw buffer accesses: the address is a uniform base, a uniform offset and a
// lane's 32-bit offset, which spares the 64-bit address arithmetic of every
// load, and a lane whose offset is past the end reads 0 and stores nothing.
typedef unsigned u32x2 __attribute__((ext_vector_type(2)));
typedef unsigned u32x4 __attribute__((ext_vector_type(4)));
typedef int i32x4 __attribute__((ext_vector_type(4)));
constexpr unsigned kNoCell = 0xFFFFFFF8u;   // an offset past every buffer's end

__device__ inline __amdgpu_buffer_rsrc_t buffer_of(const void* q, unsigned bytes)
{
    // (uniform to the compiler too: it would loop over the lanes' values otherwise)
    const uint64_t u = reinterpret_cast<uint64_t>(q);
    const unsigned lo = __builtin_amdgcn_readfirstlane(unsigned(u)), hi = __builtin_amdgcn_readfirstlane(unsigned(u >> 32));
    return __builtin_amdgcn_make_buffer_rsrc(reinterpret_cast<void*>(uint64_t(hi) << 32 | lo), 0, int(bytes), 0x00020000);
}
// aux 0x10: agent scope, a load that sees other workgroups' stores
template <typename T, int aux>
__device__ inline T buffer_load(__amdgpu_buffer_rsrc_t r, unsigned lane_off)
{
    if constexpr (aux) asm volatile("" ::: "memory");   // not to be merged with an earlier poll
    if constexpr (sizeof(T) == 4) return __builtin_bit_cast(T, __builtin_amdgcn_raw_buffer_load_b32(r, int(lane_off), 0, aux));
    else return __builtin_bit_cast(T, __builtin_amdgcn_raw_buffer_load_b64(r, int(lane_off), 0, aux));
}
template <typename T>
__device__ inline void buffer_store(__amdgpu_buffer_rsrc_t r, T v, unsigned lane_off)
{
    if constexpr (sizeof(T) == 4)
        __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned, v), r, int(lane_off), 0, 0);
    else __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(u32x2, v), r, int(lane_off), 0, 0);
}

}  // namespace m4g
