// Cross-lane steps on the VALU (DPP row moves, v_permlane16_swap / v_permlane32_swap) where a shuffle would take an LDS
// round trip (~100 cycles each, in dependent chains of three to six). The lanes a step reads must be active: the group of
// 8 or 16, or the wave.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

namespace fnkv {

// x moved by DPP control CTRL within rows of 16 lanes
template <int CTRL> __device__ __forceinline__ int32_t dpp_i(int32_t x) {
    return __builtin_amdgcn_update_dpp(0, x, CTRL, 0xf, 0xf, true);
}
template <int CTRL> __device__ __forceinline__ float dpp_f(float x) {
    return __int_as_float(dpp_i<CTRL>(__float_as_int(x)));
}
constexpr int kDppXor1 = 0xb1;        // quad_perm [1, 0, 3, 2]: lane ^ 1
constexpr int kDppXor2 = 0x4e;        // quad_perm [2, 3, 0, 1]: lane ^ 2
constexpr int kDppHalfMirror = 0x141; // 7 - lane of each 8: the other quad, once a quad's lanes agree
constexpr int kDppMirror = 0x140;     // 15 - lane of each 16: the other 8, once 8 lanes agree
constexpr int kDppRor = 0x120;        // + n: rotate the row by n (n = 8: lane ^ 8)

// max of x over each aligned group of 8 (16) lanes, in every lane of the group
__device__ __forceinline__ float max8(float x) {
    x = fmaxf(x, dpp_f<kDppXor1>(x));
    x = fmaxf(x, dpp_f<kDppXor2>(x));
    return fmaxf(x, dpp_f<kDppHalfMirror>(x));
}
__device__ __forceinline__ float max16(float x) {
    x = max8(x);
    return fmaxf(x, dpp_f<kDppMirror>(x));
}
__device__ __forceinline__ int32_t max8(int32_t x) {
    x = max(x, dpp_i<kDppXor1>(x));
    x = max(x, dpp_i<kDppXor2>(x));
    return max(x, dpp_i<kDppHalfMirror>(x));
}
// sum of x over each aligned group of 8 lanes (whole numbers)
__device__ __forceinline__ int32_t sum8(int32_t x) {
    x += dpp_i<kDppXor1>(x);
    x += dpp_i<kDppXor2>(x);
    return x + dpp_i<kDppHalfMirror>(x);
}

// the sum of x over the wave as the tree of pairs l ^ 32, l ^ 16, l ^ 8, 4, 2, 1 (each lane's bits are the shuffle
// form's: once lanes 8 (4, 2) apart agree, a rotation by 4 (2, 1) is the exchange with lane ^ 4 (2, 1))
__device__ __forceinline__ float wave_sum(float x) {
    const auto a = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    x = __uint_as_float(a[0]) + __uint_as_float(a[1]);
    const auto b = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    x = __uint_as_float(b[0]) + __uint_as_float(b[1]);
    x += dpp_f<kDppRor + 8>(x);
    x += dpp_f<kDppRor + 4>(x);
    x += dpp_f<kDppRor + 2>(x);
    return x + dpp_f<kDppRor + 1>(x);
}

// max (sum, whole numbers) of x over each half of the wave
__device__ __forceinline__ float max32(float x) {
    x = max16(x);
    const auto a = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    return fmaxf(__uint_as_float(a[0]), __uint_as_float(a[1]));
}
__device__ __forceinline__ int32_t sum32(int32_t x) {
    x = sum8(x);
    x += dpp_i<kDppMirror>(x);
    const auto a = __builtin_amdgcn_permlane16_swap(static_cast<uint32_t>(x), static_cast<uint32_t>(x), false, false);
    return static_cast<int32_t>(a[0] + a[1]);
}
// the max of x over the wave
__device__ __forceinline__ float wave_max(float x) {
    x = max32(x);
    const auto b = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    return fmaxf(__uint_as_float(b[0]), __uint_as_float(b[1]));
}

} // namespace fnkv
