// Float-math products of many rows with at most 128 inputs, in Trit's 16-lane
// sum order (gemv_float.hip), the same bits. A code object of its own: the
// unrolled chains of every width and kind, with and without the GELU, are 230 KB
// that a process which never runs such a layer does not load (a code object
// loads whole with its first kernel, about 1.8 us a KB).
#include "float_weights.h"

#include <type_traits>

namespace trit {
namespace {

constexpr int THREADS = 256;

// Many input rows of a layer with few inputs (k <= 16 S; an audio stem's
// first convolution): block (x, y) takes 256 output columns and RB input
// rows; a thread holds its column's 16 lane chains (S steps each) in
// registers and runs them over the rows, then the tree16 order of the
// small-batch kernels, so every row gets their bits.
template <int K, int S, bool GELU>
__global__ __launch_bounds__(THREADS) void float_rows_kernel(const typename WT<K>::E* __restrict__ w,
                                                             const float* __restrict__ scales,
                                                             const float* __restrict__ bias, int n, int k, GemvArgs a) {
    constexpr int RB = 64;
    const int col = blockIdx.x * THREADS + (int)threadIdx.x;
    if (col >= n) return;
    const int s_count = chain_steps(k);  // <= S
    float wr[16][S];
#pragma unroll
    for (int i = 0; i < 16; ++i)
#pragma unroll
        for (int st = 0; st < S; ++st)
            wr[i][st] = st < s_count ? widen1<K>(w + ((size_t)col * 16 + i) * s_count,
                                                 scales ? scales + (size_t)col * (k / 32) : nullptr, st)
                                     : 0.0f;
    const int f1 = min(a.m, (int)(blockIdx.y + 1) * RB);
    for (int f = blockIdx.y * RB; f < f1; ++f) {
        const float* xf = a.x + (size_t)f * k;
        float l[16];
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            float acc = 0.0f;
#pragma unroll
            for (int st = 0; st < S; ++st) {
                const int kk = 16 * st + i;
                acc = __builtin_fmaf(kk < k ? xf[kk] : 0.0f, wr[i][st], acc);
            }
            l[i] = acc;
        }
        float h[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) h[i] = l[i] + l[i + 8];
        float v[1] = {((h[0] + h[4]) + (h[2] + h[6])) + ((h[1] + h[5]) + (h[3] + h[7]))};
        if constexpr (GELU) {
            finish_outputs<true>(v, bias, {col}, a.relu);
            const size_t at = (size_t)f * n + col;
            a.y[at] = a.epilogue == EPI_RESIDUAL ? a.residual[at] + v[0] : v[0];
        } else {
            store_out(a, bias, n, f, col, v[0]);
        }
    }
}

}  // namespace

bool gemm_float_supported(const Layer& L, const GemvArgs& a) {
    return float_kind(L.kind) && L.k <= 128 && a.m >= 1 && !a.norm_w && a.epilogue != EPI_SILU_PAIR;
}

void gemm_float(const Layer& L, const GemvArgs& a, hipStream_t s) {
    if (!gemm_float_supported(L, a)) fail("float rows: a float-math layer of k <= 128, no prologue or pair");
    auto go = [&](auto K_, auto S_) {
        constexpr int K = decltype(K_)::value, S = decltype(S_)::value;
        using E = typename WT<K>::E;
        const dim3 grid((L.n + THREADS - 1) / THREADS, (a.m + 63) / 64);
        launch_timed(a, a.gelu ? float_rows_kernel<K, S, true> : float_rows_kernel<K, S, false>, grid, dim3(THREADS), 0,
                     s, L.codes.as<E>(), K == WK_Q8 ? L.scales.as<float>() : nullptr, L.bias.as<float>(), L.n, L.k, a);
    };
    auto by_steps = [&](auto K_) {
        const int steps = chain_steps(L.k);
        if (steps <= 1) go(K_, std::integral_constant<int, 1>{});
        else if (steps <= 2) go(K_, std::integral_constant<int, 2>{});
        else if (steps <= 4) go(K_, std::integral_constant<int, 4>{});
        else go(K_, std::integral_constant<int, 8>{});
    };
    switch (L.kind) {
        case F16: by_steps(std::integral_constant<int, WK_F16>{}); break;
        case F32: by_steps(std::integral_constant<int, WK_F32>{}); break;
        default: by_steps(std::integral_constant<int, WK_Q8>{}); break;
    }
    TRIT_HIP(hipGetLastError());
}

}  // namespace trit
