// Reductions over the 64 lanes of a wave, or over aligned groups of 16 of them,
// that every lane of the group ends with.
//
// Six dependent steps, each an add of a neighbour's value.  Through __shfl_xor a
// step is an LDS permute and its wait, which the kernels of the one-token step (3
// to 6 us each, all latency) pay up to a dozen times in their chain.  Here lanes
// 1, 2, 4 and 8 apart meet through the DPP operand of the add itself, and rows 16
// and 32 apart through the lane swaps of gfx950, without LDS: a token of GPT-2
// small (B = 1, 512 keys, 62 launches) went from 356 to 336 us.  Kernels bound by
// bandwidth (LayerNorm, the loss) measure the same either way.
#pragma once

#include <hip/hip_runtime.h>

namespace gptc {

template <int kCtrl>
__device__ __forceinline__ float dpp_of(float v) {
    const int i = __float_as_int(v);
    return __int_as_float(__builtin_amdgcn_update_dpp(i, i, kCtrl, 0xf, 0xf, true));
}

constexpr int kDppXor1 = 0xb1;         // quad_perm 1 0 3 2
constexpr int kDppXor2 = 0x4e;         // quad_perm 2 3 0 1
constexpr int kDppHalfMirror = 0x141;  // lane 7 - l of the 8: the other quad
constexpr int kDppMirror = 0x140;      // lane 15 - l of the row: the other half

// Sum and max over each row of 16 lanes.  After the steps 1 and 2 apart a quad
// holds one value, so the mirrored half row is the quad 4 apart, and after that
// the mirrored row the half 8 apart.
__device__ __forceinline__ float row16_sum(float v) {
    v += dpp_of<kDppXor1>(v);
    v += dpp_of<kDppXor2>(v);
    v += dpp_of<kDppHalfMirror>(v);
    return v + dpp_of<kDppMirror>(v);
}

__device__ __forceinline__ float row16_max(float v) {
    v = fmaxf(v, dpp_of<kDppXor1>(v));
    v = fmaxf(v, dpp_of<kDppXor2>(v));
    v = fmaxf(v, dpp_of<kDppHalfMirror>(v));
    return fmaxf(v, dpp_of<kDppMirror>(v));
}

// Max and sum over the four lanes l % 16 + {0, 16, 32, 48} (one query of a
// 16 x 16 accumulator), every lane receiving the result.  gfx950's
// v_permlane32_swap / v_permlane16_swap exchange lane halves / 16-lane rows
// in the VALU: with both operands equal to x, the two results hold x at the
// lane and at its partner (l ^ 32, then l ^ 16), in some order.
__device__ __forceinline__ float max4_rows(float x) {
    const auto h = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    const float y = fmaxf(__uint_as_float(h[0]), __uint_as_float(h[1]));
    const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(y), __float_as_uint(y), false, false);
    return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}

__device__ __forceinline__ float sum4_rows(float x) {
    const auto h = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    const float y = __uint_as_float(h[0]) + __uint_as_float(h[1]);
    const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(y), __float_as_uint(y), false, false);
    return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}

__device__ __forceinline__ float wave_sum(float v) { return sum4_rows(row16_sum(v)); }
__device__ __forceinline__ float wave_max(float v) { return max4_rows(row16_max(v)); }

}  // namespace gptc
