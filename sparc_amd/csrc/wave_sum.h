// Sums over a wavefront without LDS: lane swaps and rotations of gfx950.
#ifndef SPARC_AMD_WAVE_SUM_H
#define SPARC_AMD_WAVE_SUM_H

#include <hip/hip_runtime.h>

// Sums of four values over the wave: in the 16 lanes of row g, the sum of
// s[g].  Two half-wave swaps, one 16-lane swap (each adds two values' halves
// side by side), then rotations within the row: a third of the operations of
// four wave_sum_f64.
__device__ __forceinline__ double swap_add(double a, double b, bool half)
{
    const unsigned long long ua = __double_as_longlong(a), ub = __double_as_longlong(b);
    unsigned int lo[2], hi[2];
    if (half) {
        const auto l = __builtin_amdgcn_permlane32_swap((unsigned)ua, (unsigned)ub, false, false);
        const auto h = __builtin_amdgcn_permlane32_swap((unsigned)(ua >> 32), (unsigned)(ub >> 32), false, false);
        lo[0] = l[0]; lo[1] = l[1]; hi[0] = h[0]; hi[1] = h[1];
    } else {
        const auto l = __builtin_amdgcn_permlane16_swap((unsigned)ua, (unsigned)ub, false, false);
        const auto h = __builtin_amdgcn_permlane16_swap((unsigned)(ua >> 32), (unsigned)(ub >> 32), false, false);
        lo[0] = l[0]; lo[1] = l[1]; hi[0] = h[0]; hi[1] = h[1];
    }
    return __longlong_as_double((long long)(((unsigned long long)hi[0] << 32) | lo[0])) +
           __longlong_as_double((long long)(((unsigned long long)hi[1] << 32) | lo[1]));
}

template <int N>
__device__ __forceinline__ double row_ror_f64(double v)
{
    const long long b = __double_as_longlong(v);
    const int lo = __builtin_amdgcn_update_dpp(0, (int)(b & 0xffffffff), 0x120 + N, 0xf, 0xf, true);
    const int hi = __builtin_amdgcn_update_dpp(0, (int)(b >> 32), 0x120 + N, 0xf, 0xf, true);
    return __longlong_as_double(((long long)hi << 32) | (unsigned int)lo);
}

__device__ __forceinline__ double rows4_sum(double s0, double s1, double s2, double s3)
{
    // lanes 0-31 / 32-63 hold s0 / s2 and s1 / s3, then rows 0..3 hold s0..s3
    double v = swap_add(swap_add(s0, s2, true), swap_add(s1, s3, true), false);
    v += row_ror_f64<8>(v);
    v += row_ror_f64<4>(v);
    v += row_ror_f64<2>(v);
    v += row_ror_f64<1>(v);
    return v;
}

#endif
