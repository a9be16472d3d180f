// proposal.h -- the proposed spin of an attempt, looked up: the new spin is the
// old one (-1, 0, 1) plus the step of the random word (+1 below 2^31, else -1),
// wrapped into -1..1.  The six cases are bytes of two dwords, taken with one
// v_perm_b32 per quantity (selector bytes 0-3 take the second dword's bytes,
// 4-7 the first's, 0x0c is zero).
#pragma once
#include <stdint.h>
#include <hip/hip_runtime.h>

namespace muca {

// old + 1, + 4 for a step down
__device__ __forceinline__ uint32_t proposal_index(int32_t old_s, uint32_t r3)
{
    return (uint32_t)old_s + 0x0c0c0c01u + ((r3 >> 29) & 4u);
}
// minus the spin change
__device__ __forceinline__ int32_t proposal_mds(uint32_t at)
{
    return (int32_t)(int8_t)__builtin_amdgcn_perm(0x000101feu, 0x0002ffffu, at);
}
// the change of D = sum s^2
__device__ __forceinline__ int32_t proposal_ddel(uint32_t at)
{
    return (int32_t)(int8_t)__builtin_amdgcn_perm(0x00ff0100u, 0x000001ffu, at);
}
// the new spin's byte
__device__ __forceinline__ uint32_t proposal_new(uint32_t at)
{
    return __builtin_amdgcn_perm(0x0000ff01u, 0x00ff0100u, at);
}

}  // namespace muca
