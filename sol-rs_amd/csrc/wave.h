// wave.h -- reductions over a wave64 or over groups of 8 lanes, on DPP (one
// VALU instruction per step; __shfl_xor goes through the LDS pipe).
// Every lane of the wave must be active.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace solhip {

// v from the lane that CTRL names; lanes without a source (and rows outside
// ROWS) get `old`
template <int CTRL, int ROWS = 0xF>
__device__ __forceinline__ uint32_t dpp(uint32_t old, uint32_t v)
{
    return (uint32_t)__builtin_amdgcn_update_dpp((int)old, (int)v, CTRL, ROWS, 0xF, false);
}

// floats as unsigned integers of the same order
__device__ __forceinline__ uint32_t f2ord(float f)
{
    uint32_t b = __float_as_uint(f);
    return (b & 0x80000000u) ? ~b : (b | 0x80000000u);
}
__device__ __forceinline__ float ord2f(uint32_t u)
{
    return __uint_as_float((u & 0x80000000u) ? (u & 0x7FFFFFFFu) : ~u);
}

// groups of 8 lanes: lanes xor 1, xor 2 (quad_perm), then the two quads
// (row_half_mirror); every lane gets its group's result
template <class Op>
__device__ __forceinline__ uint32_t group8(uint32_t v, Op op)
{
    v = op(v, dpp<0xB1>(v, v));
    v = op(v, dpp<0x4E>(v, v));
    return op(v, dpp<0x141>(v, v));
}
__device__ __forceinline__ uint32_t group8_min(uint32_t v)
{
    return group8(v, [](uint32_t a, uint32_t b) { return min(a, b); });
}
__device__ __forceinline__ uint32_t group8_max(uint32_t v)
{
    return group8(v, [](uint32_t a, uint32_t b) { return max(a, b); });
}
__device__ __forceinline__ float group8_fmin(float v)
{
    return __uint_as_float(group8(__float_as_uint(v), [](uint32_t a, uint32_t b) {
        return __float_as_uint(fminf(__uint_as_float(a), __uint_as_float(b)));
    }));
}
__device__ __forceinline__ float group8_fmax(float v)
{
    return __uint_as_float(group8(__float_as_uint(v), [](uint32_t a, uint32_t b) {
        return __float_as_uint(fmaxf(__uint_as_float(a), __uint_as_float(b)));
    }));
}

// whole wave: rows of 16 by row_shr, then across rows by row_bcast; the result
// is in lane 63 and returned to every lane
template <class Op>
__device__ __forceinline__ uint32_t wave_reduce(uint32_t v, uint32_t identity, Op op)
{
    v = op(v, dpp<0x111>(identity, v));
    v = op(v, dpp<0x112>(identity, v));
    v = op(v, dpp<0x114>(identity, v));
    v = op(v, dpp<0x118>(identity, v));
    v = op(v, dpp<0x142, 0xA>(identity, v));
    v = op(v, dpp<0x143, 0xC>(identity, v));
    return (uint32_t)__builtin_amdgcn_readlane((int)v, 63);
}
__device__ __forceinline__ uint32_t wave_min(uint32_t v)
{
    return wave_reduce(v, 0xFFFFFFFFu, [](uint32_t a, uint32_t b) { return min(a, b); });
}
__device__ __forceinline__ uint32_t wave_max(uint32_t v)
{
    return wave_reduce(v, 0u, [](uint32_t a, uint32_t b) { return max(a, b); });
}

// inclusive scan within each half of 32 lanes
template <class Op>
__device__ __forceinline__ uint32_t half_scan(uint32_t v, uint32_t identity, Op op)
{
    v = op(v, dpp<0x111>(identity, v));
    v = op(v, dpp<0x112>(identity, v));
    v = op(v, dpp<0x114>(identity, v));
    v = op(v, dpp<0x118>(identity, v));
    return op(v, dpp<0x142, 0xA>(identity, v));
}

// orders this wave's LDS accesses (no other wave is involved)
__device__ __forceinline__ void wave_lds_sync()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

}  // namespace solhip
