// What the float-math products share (gemv_float.hip, float_rows.hip,
// gemm_float.hip): the weight kinds' elements in the lane-chain layout, their
// widening, an output's store.
#pragma once

#include "device.h"
#include "internal.h"

namespace trit {
namespace {

// Weight kinds: element type and elements per 16-byte unit.
enum WKind { WK_F16, WK_F32, WK_Q8 };
template <int K>
struct WT;
template <>
struct WT<WK_F16> {
    using E = uint16_t;
    static constexpr int PER = 8;
};
template <>
struct WT<WK_F32> {
    using E = float;
    static constexpr int PER = 4;
};
template <>
struct WT<WK_Q8> {
    using E = int8_t;
    static constexpr int PER = 16;
};

// One element of a chain, widened: w[s] (f16, f32) or f32(code) * scale.
template <int K>
__device__ __forceinline__ float widen1(const typename WT<K>::E* chain, const float* row_scales, int s) {
    if constexpr (K == WK_F16) return f16_to_f32(chain[s]);
    else if constexpr (K == WK_F32) return chain[s];
    else return (float)chain[s] * row_scales[s >> 1];
}

__device__ __forceinline__ void store_out(const GemvArgs& a, const float* __restrict__ bias, int n, int f, int row,
                                          float v) {
    if (bias) v = v + bias[row];
    if (a.relu) v = __builtin_fmaxf(v, 0.0f);
    const size_t at = (size_t)f * n + row;
    a.y[at] = a.epilogue == EPI_RESIDUAL ? a.residual[at] + v : v;
}

}  // namespace
}  // namespace trit
