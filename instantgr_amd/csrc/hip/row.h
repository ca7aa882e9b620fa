// Data movement inside a wave's 16-lane rows (DPP: no LDS, no wait), and
// compile-time loops, for kernels that keep one layer per lane of a row.
// Every lane of the wave must be active where these are called.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>

namespace igr_dev {

// f(integral_constant 0 .. N - 1), fully unrolled.
template <int N, int I = 0, class F>
__device__ __forceinline__ void unrolled(F f) {
    if constexpr (I < N) {
        f(std::integral_constant<int, I>{});
        unrolled<N, I + 1>(f);
    }
}

// Value of lane N of the caller's row.
template <int N>
__device__ __forceinline__ int row_bcast(int v) {
    return __builtin_amdgcn_mov_dpp(v, 0x150 + N, 0xf, 0xf, false);
}
template <int N>
__device__ __forceinline__ float row_bcast(float v) {
    return __int_as_float(row_bcast<N>(__float_as_int(v)));
}
template <int N>
__device__ __forceinline__ double row_bcast(double v) {
    const int64_t b = __double_as_longlong(v);
    const int lo = row_bcast<N>((int)b), hi = row_bcast<N>((int)(b >> 32));
    return __longlong_as_double(((int64_t)hi << 32) | (uint32_t)lo);
}

// Value of the lane D above in the caller's row, +inf past its end.
template <int D>
__device__ __forceinline__ double row_above(double v) {
    const int64_t b = __double_as_longlong(v);
    const int lo = __builtin_amdgcn_update_dpp(0, (int)b, 0x100 + D, 0xf, 0xf, false);
    const int hi = __builtin_amdgcn_update_dpp(0x7ff00000, (int)(b >> 32), 0x100 + D, 0xf, 0xf, false);
    return __longlong_as_double(((int64_t)hi << 32) | (uint32_t)lo);
}

} // namespace igr_dev
