// bs_wave.hpp -- sums over the lanes of a wave, in a fixed order, by DPP moves
// and lane swaps: three VALU instructions a step.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace bs {

// x moved across lanes by a DPP control; lanes it does not reach, and rows
// outside `rows`, give 0.
template <int kControl, int kRows>
__device__ __forceinline__ double dpp(double x) {
    const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(x), kControl, kRows, 0xf, true);
    const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(x), kControl, kRows, 0xf, true);
    return __hiloint2double(hi, lo);
}

// The sums of the four rows of 16 lanes, in lanes 15, 31, 47 and 63 (shifts right
// by 1, 2, 4, 8).
__device__ __forceinline__ double row_sums(double x) {
    x += dpp<0x111, 0xf>(x);
    x += dpp<0x112, 0xf>(x);
    x += dpp<0x114, 0xf>(x);
    x += dpp<0x118, 0xf>(x);
    return x;
}

// The sums of lanes 0-31 in lane 31 and of lanes 32-63 in lane 63: within rows of
// 16 lanes (shifts right by 1, 2, 4, 8), then row totals into the next row
// (broadcast of lane 15).
__device__ __forceinline__ double half_wave_sum(double x) {
    x = row_sums(x);
    x += dpp<0x142, 0xa>(x);
    return x;
}

// The wave's sum, in every lane: lane 31's half into the upper one's (broadcast).
// Through LDS (__shfl_xor) the five folds of a portfolio wave cost as much as two
// of its options.
__device__ __forceinline__ double wave_sum(double x) {
    x = half_wave_sum(x);
    x += dpp<0x143, 0xc>(x);
    return __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(x), 63),
                            __builtin_amdgcn_readlane(__double2loint(x), 63));
}

// a and b, each the halves of two quantities (swap_halves_add), folded into a row
// each: row 0 gets a of rows 0 and 1 added, row 1 the same of b, rows 2 and 3
// those of rows 2 and 3.
__device__ __forceinline__ double swap_rows_add(double a, double b) {
    const auto lo = __builtin_amdgcn_permlane16_swap((uint32_t)__double2loint(a),
                                                     (uint32_t)__double2loint(b), false, false);
    const auto hi = __builtin_amdgcn_permlane16_swap((uint32_t)__double2hiint(a),
                                                     (uint32_t)__double2hiint(b), false, false);
    return __hiloint2double((int)hi[0], (int)lo[0]) + __hiloint2double((int)hi[1], (int)lo[1]);
}

// Two quantities folded into half a wave each: lanes 0-31 get a of lanes l and
// l + 32 added, lanes 32-63 the same of b.
__device__ __forceinline__ double swap_halves_add(double a, double b) {
    const auto lo = __builtin_amdgcn_permlane32_swap((uint32_t)__double2loint(a),
                                                     (uint32_t)__double2loint(b), false, false);
    const auto hi = __builtin_amdgcn_permlane32_swap((uint32_t)__double2hiint(a),
                                                     (uint32_t)__double2hiint(b), false, false);
    return __hiloint2double((int)hi[0], (int)lo[0]) + __hiloint2double((int)hi[1], (int)lo[1]);
}

}  // namespace bs
