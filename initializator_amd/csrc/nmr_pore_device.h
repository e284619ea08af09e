// nmr_pore_device.h -- device functions shared by the kernels over the list of
// the pores (nmr_pores.hip, nmr_pore_blocks.hip).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace nmr {

// Values that the compiler must have at this point: it would otherwise sink
// the load behind a select (of a base, of the neighbours' values) into a
// branch, one dependent wait each.
template <typename T>
__device__ __forceinline__ void have_s(T& x)
{
    asm volatile("" : "+s"(x));
}
__device__ __forceinline__ void have_v(float& x) { asm volatile("" : "+v"(x)); }

// State of slot i, NC floats per slot.  Byte offsets stay below 4 GiB, so an
// access is a scalar base plus a 32-bit offset.
template <int NC>
struct VecOf;
template <>
struct VecOf<1> {
    typedef float type __attribute__((ext_vector_type(1)));
};
template <>
struct VecOf<2> {
    typedef float type __attribute__((ext_vector_type(2)));
};
template <>
struct VecOf<3> {
    typedef float type __attribute__((ext_vector_type(3), aligned(4)));
};
template <int NC>
using Vec = typename VecOf<NC>::type;

template <int NC>
__device__ __forceinline__ void stm(float* base, uint32_t i, const Vec<NC>& v)
{
    *reinterpret_cast<Vec<NC>*>(reinterpret_cast<char*>(base) + i * (uint32_t)(4 * NC)) = v;
}
template <typename T>
__device__ __forceinline__ T ldw(const T* base, uint32_t i)
{
    return *reinterpret_cast<const T*>(reinterpret_cast<const char*>(base) + i * (uint32_t)sizeof(T));
}

// A value at byte offset o of an array.
template <typename T>
__device__ __forceinline__ T at_byte(const void* base, uint32_t o)
{
    return *reinterpret_cast<const T*>(reinterpret_cast<const char*>(base) + o);
}

// v of another lane by a DPP move of both halves (0 where the move has no source).
template <int CTRL, int ROWS>
__device__ __forceinline__ double dpp_add(double v)
{
    const uint64_t b = (uint64_t)__double_as_longlong(v);
    const uint32_t lo = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(uint32_t)b, CTRL, ROWS, 0xf, false);
    const uint32_t hi = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(uint32_t)(b >> 32), CTRL, ROWS, 0xf, false);
    return v + __longlong_as_double((long long)(((uint64_t)hi << 32) | lo));
}

// Sum over the wavefront, in lane 63: within rows of 16 lanes by shifts,
// then across the rows by broadcasts -- register moves, where a shuffle
// through LDS costs a round trip each.
__device__ __forceinline__ double wave_sum(double v)
{
    v = dpp_add<0x111, 0xf>(v); // row_shr:1
    v = dpp_add<0x112, 0xf>(v); // row_shr:2
    v = dpp_add<0x114, 0xf>(v); // row_shr:4
    v = dpp_add<0x118, 0xf>(v); // row_shr:8
    v = dpp_add<0x142, 0xa>(v); // row_bcast:15 into rows 1 and 3
    v = dpp_add<0x143, 0xc>(v); // row_bcast:31 into rows 2 and 3
    return v;
}

// max(v, 0) and min(v, 0) (0 for a NaN) without the canonicalisation that
// fmaxf adds for signalling NaNs, which no loaded sum is.
__device__ __forceinline__ float pos(float v)
{
    float r;
    asm("v_max_f32 %0, 0, %1" : "=v"(r) : "v"(v));
    return r;
}
__device__ __forceinline__ float neg(float v)
{
    float r;
    asm("v_min_f32 %0, 0, %1" : "=v"(r) : "v"(v));
    return r;
}

} // namespace nmr
