// Workgroup Sklansky scan reproducing the reference's association order
// (src/graph.hpp:412-417): over a virtual array s[0..n), level d adds to every
// element whose index has bit d set the last element of the preceding 2^d
// block.  Thread t of the workgroup holds elements t*K .. t*K+K-1 in
// registers (K a power of two), so levels below log2(K) run inside a thread,
// the next six levels across the lanes of a wave and the rest across waves
// through LDS.  Each element receives the same additions in the same level
// order as the sequential loop, so floating-point results are bit-identical to
// it.  Elements at or beyond n never influence those below n.
//
// The lanes' levels move values with DPP (a level's source is lane 2^d - 1 of
// each block of 2^(d+1) lanes: quad permutes, row broadcasts with bank masks,
// then the row broadcasts that cross rows), so no level waits for the LDS.
// The wave totals are read once, one per lane, and their levels run the same
// way in every wave, which picks its own addends by lane reads: one barrier.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace igr_dev {

template <int CTRL, int ROWS, int BANKS>
__device__ __forceinline__ int dpp_move(int old, int v) {
    return __builtin_amdgcn_update_dpp(old, v, CTRL, ROWS, BANKS, false);
}
template <int CTRL, int ROWS, int BANKS>
__device__ __forceinline__ float dpp_move(float old, float v) {
    return __int_as_float(dpp_move<CTRL, ROWS, BANKS>(__float_as_int(old), __float_as_int(v)));
}
template <int CTRL, int ROWS, int BANKS>
__device__ __forceinline__ double dpp_move(double old, double v) {
    const int64_t o = __double_as_longlong(old), b = __double_as_longlong(v);
    const int lo = dpp_move<CTRL, ROWS, BANKS>((int)o, (int)b);
    const int hi = dpp_move<CTRL, ROWS, BANKS>((int)(o >> 32), (int)(b >> 32));
    return __longlong_as_double(((int64_t)hi << 32) | (uint32_t)lo);
}

// Level D (0 .. 5) of the scan across lanes: for every lane with bit D set,
// the value of the last lane of the preceding 2^D block.
template <int D, typename T>
__device__ __forceinline__ T sklansky_source(T v) {
    if constexpr (D == 0) return dpp_move<0xA0, 0xf, 0xf>(v, v);          // quad lanes 0 0 2 2
    else if constexpr (D == 1) return dpp_move<0x54, 0xf, 0xf>(v, v);     // quad lanes . . 1 1
    else if constexpr (D == 2)                                            // lane 3 to 4..7, lane 11 to 12..15
        return dpp_move<0x150 + 11, 0xf, 0x8>(dpp_move<0x150 + 3, 0xf, 0x2>(v, v), v);
    else if constexpr (D == 3) return dpp_move<0x150 + 7, 0xf, 0xc>(v, v);   // lane 7 to 8..15
    else if constexpr (D == 4) return dpp_move<0x142, 0xa, 0xf>(v, v);    // lane 15 of a row to the next
    else return dpp_move<0x143, 0xc, 0xf>(v, v);                          // lane 31 to rows 2 and 3
}

__device__ __forceinline__ int lane_read(int v, int lane) { return __builtin_amdgcn_readlane(v, lane); }
__device__ __forceinline__ float lane_read(float v, int lane) { return __int_as_float(lane_read(__float_as_int(v), lane)); }
__device__ __forceinline__ double lane_read(double v, int lane) {
    const int64_t b = __double_as_longlong(v);
    const int lo = lane_read((int)b, lane), hi = lane_read((int)(b >> 32), lane);
    return __longlong_as_double(((int64_t)hi << 32) | (uint32_t)lo);
}

template <int D, typename T, int K>
__device__ __forceinline__ void sklansky_level(T (&s)[K]) {
    const T v = sklansky_source<D>(s[K - 1]);
    if (threadIdx.x >> D & 1) {
#pragma unroll
        for (int j = 0; j < K; j++) s[j] += v;
    }
}
template <int B, typename T, int K>
__device__ __forceinline__ void sklansky_wave_level(T (&s)[K], T& w, int wave) {
    const T add = lane_read(w, ((wave >> B) << B) > 0 ? ((wave >> B) << B) - 1 : 0);
    if (wave >> B & 1) {
#pragma unroll
        for (int j = 0; j < K; j++) s[j] += add;
    }
    const T v = sklansky_source<B>(w);
    if (threadIdx.x >> B & 1) w += v;
}

// lds_tot: 16 entries that no other exchange of the kernel uses between the
// barriers around this call (the one inside orders the totals; a second scan
// on the same entries needs a barrier before it).
template <typename T, int K>
__device__ __forceinline__ void block_sklansky_rt(T (&s)[K], T* lds_tot, int nw) {
#pragma unroll
    for (int d = 0; (1 << d) < K; d++) {
#pragma unroll
        for (int j = 0; j < K; j++)
            if (j >> d & 1) s[j] += s[(j >> d << d) - 1];
    }
    sklansky_level<0>(s);
    sklansky_level<1>(s);
    sklansky_level<2>(s);
    sklansky_level<3>(s);
    sklansky_level<4>(s);
    sklansky_level<5>(s);
    if (nw > 1) {
        const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
        if (lane == 63) lds_tot[wave] = s[K - 1];
        __syncthreads();
        T w = (lane & 15) < nw ? lds_tot[lane & 15] : T(0);
        sklansky_wave_level<0>(s, w, wave);
        if (nw > 2) sklansky_wave_level<1>(s, w, wave);
        if (nw > 4) sklansky_wave_level<2>(s, w, wave);
        if (nw > 8) sklansky_wave_level<3>(s, w, wave);
    }
}

} // namespace igr_dev
