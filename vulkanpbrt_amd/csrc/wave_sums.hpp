// Sums over a wave of 64 lanes of several values at once.
//
// A butterfly (v += shuffle(v, xor 32), ... xor 1) through the LDS pipe costs two
// operations per value and step.  Here the lanes hold different values from the first
// step on: v_permlane32_swap / v_permlane16_swap exchange half a register with another
// value's, so xor 32 and xor 16 cost one swap and one add per two values, and the steps
// inside a row of 16 lanes are DPP adds.  Every sum is the same binary tree over the
// same lanes as the butterfly from xor 32 down to xor 1.
#pragma once

#include <hip/hip_runtime.h>

namespace pbrt {

// LDS written by some lanes of a wave and then read by others of the same wave, or read
// and then written again: the hardware completes a wave's LDS operations in order, and the
// fences keep the compiler from moving them past each other.
__device__ __forceinline__ void wave_lds_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

__device__ __forceinline__ float swap_add32(float a, float b) {
    // lanes 0..31: a[l] + a[l ^ 32]; lanes 32..63: b[l] + b[l ^ 32]
    const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(a), __float_as_uint(b), false, false);
    return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}
__device__ __forceinline__ float swap_add16(float a, float b) {
    // rows 0, 2: a[l] + a[l ^ 16]; rows 1, 3: b[l] + b[l ^ 16]
    const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(a), __float_as_uint(b), false, false);
    return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}
template <int kCtrl>
__device__ __forceinline__ float dpp_add(float v) {
    return v + __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), kCtrl, 0xF, 0xF, true));
}
// four values by row: row r of the result holds value r's xor-32 and xor-16 steps
__device__ __forceinline__ float rows_of(float s0, float s1, float s2, float s3) {
    return swap_add16(swap_add32(s0, s2), swap_add32(s1, s3));
}
// the xor-8 and xor-4 steps: each lane adds its row's lane l ^ 8, then (the row being
// 8-periodic) the one four further, which holds the value of l ^ 4
__device__ __forceinline__ float row_steps84(float v) { return dpp_add<0x124>(dpp_add<0x128>(v)); }  // row_ror 8, 4
// the xor-2 and xor-1 steps inside each quartet of lanes
__device__ __forceinline__ float quad_steps21(float v) { return dpp_add<0xB1>(dpp_add<0x4E>(v)); }  // quad_perm
// one value: its sum on every lane
__device__ __forceinline__ float wave_sum(float v) {
    v = swap_add32(v, v);
    v = swap_add16(v, v);
    return quad_steps21(row_steps84(v));
}
// the registers' own values by lane quartet (bank = (lane / 4) % 4)
__device__ __forceinline__ float by_bank(int bank, float s0, float s1, float s2, float s3) {
    const float lo = (bank & 1) ? s1 : s0, hi = (bank & 1) ? s3 : s2;
    return (bank & 2) ? hi : lo;
}

}  // namespace pbrt
