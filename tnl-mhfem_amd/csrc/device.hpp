// device.hpp -- device helpers shared by the Krylov translation units:
// wavefront sums, and values handed from one work-group to another while both
// run (a value is its own flag: it is there once it no longer holds a
// signalling-NaN payload that arithmetic never produces).
#pragma once

#include <hip/hip_runtime.h>

namespace mhfem {

__device__ __forceinline__ double wave_sum(double v)
{
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
    return v;
}

// Sums over the wavefront of several values at once.  Each step adds the two
// halves of the lanes while handing one half to the other value of a pair
// (v_permlane32_swap, v_permlane16_swap), so that ND sums cost little more
// than one; the last 16 lanes are summed with row rotations.  No LDS is
// touched.  sums_wave<ND> leaves dot d in the lanes with
// lane / (64 / ND) == d.
__device__ __forceinline__ double swap_add32(double a, double b)
{
    const unsigned long long x = __builtin_bit_cast(unsigned long long, a), y = __builtin_bit_cast(unsigned long long, b);
    const auto lo = __builtin_amdgcn_permlane32_swap((unsigned)x, (unsigned)y, false, false);
    const auto hi = __builtin_amdgcn_permlane32_swap((unsigned)(x >> 32), (unsigned)(y >> 32), false, false);
    return __builtin_bit_cast(double, (unsigned long long)hi[0] << 32 | lo[0]) +
           __builtin_bit_cast(double, (unsigned long long)hi[1] << 32 | lo[1]);
}
__device__ __forceinline__ double swap_add16(double a, double b)
{
    const unsigned long long x = __builtin_bit_cast(unsigned long long, a), y = __builtin_bit_cast(unsigned long long, b);
    const auto lo = __builtin_amdgcn_permlane16_swap((unsigned)x, (unsigned)y, false, false);
    const auto hi = __builtin_amdgcn_permlane16_swap((unsigned)(x >> 32), (unsigned)(y >> 32), false, false);
    return __builtin_bit_cast(double, (unsigned long long)hi[0] << 32 | lo[0]) +
           __builtin_bit_cast(double, (unsigned long long)hi[1] << 32 | lo[1]);
}
template <int ROR>
__device__ __forceinline__ double rotate_add(double a)
{
    const unsigned long long x = __builtin_bit_cast(unsigned long long, a);
    const unsigned lo = __builtin_amdgcn_update_dpp(0, (int)(unsigned)x, 0x120 + ROR, 0xf, 0xf, false);
    const unsigned hi = __builtin_amdgcn_update_dpp(0, (int)(unsigned)(x >> 32), 0x120 + ROR, 0xf, 0xf, false);
    return a + __builtin_bit_cast(double, (unsigned long long)hi << 32 | lo);
}
template <int ND>
__device__ __forceinline__ double sums_wave(const double (&v)[ND])
{
    static_assert(ND == 1 || ND == 2 || ND == 4);
    double t;
    if constexpr (ND == 4) t = swap_add16(swap_add32(v[0], v[2]), swap_add32(v[1], v[3]));
    else if constexpr (ND == 2) {
        const double u = swap_add32(v[0], v[1]);
        t = swap_add16(u, u);
    } else {
        const double u = swap_add32(v[0], v[0]);
        t = swap_add16(u, u);
    }
    return rotate_add<1>(rotate_add<2>(rotate_add<4>(rotate_add<8>(t))));
}

template <typename T>
struct SentinelBits;
template <>
struct SentinelBits<double> {
    using U = unsigned long long;
    static constexpr U bits = 0x7FF4A5A5A5A5A5A5ull;
};
template <>
struct SentinelBits<float> {
    using U = unsigned int;
    static constexpr U bits = 0x7FA5A5A5u;
};
template <typename T>
__device__ __forceinline__ bool is_sentinel(T v)
{
    return __builtin_bit_cast(typename SentinelBits<T>::U, v) == SentinelBits<T>::bits;
}
template <typename T>
__device__ __forceinline__ T sentinel_value()
{
    return __builtin_bit_cast(T, SentinelBits<T>::bits);
}
template <typename T>
__device__ __forceinline__ T coherent_load(const T *p)
{
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
template <typename T>
__device__ __forceinline__ void coherent_store(T *p, T v)
{
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
template <typename T>
__device__ __forceinline__ T lds_load(const T *p)
{
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}
template <typename T>
__device__ __forceinline__ void lds_store(T *p, T v)
{
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}

}  // namespace mhfem
