// Float-math products (f16, f32 and int8-storage weights) of many rows on
// the f32 matrix cores, in Trit's 16-lane sum order, bit for bit the
// small-batch kernels' results (gemv_float.hip; src/cpu/fgemm.rs:413-455):
// output (row, col) is the 16-lane tree over the lane chains
// acc_i = fma(x[16 s + i], w[16 s + i], acc_i), s in order from +0.
//
// v_mfma_f32_16x16x4_f32 is that chain: each of its outputs is four fused
// multiply-adds in k order onto the accumulator, every one rounded to
// nearest even with subnormals kept (checked on the device against fmaf
// over wide exponent ranges, subnormal inputs and results: no difference in
// 51200 outputs a range; the reverse k order differs). So lane chain i of a
// 16 x 16 tile is one MFMA sequence over its steps s, four a time, and the
// sixteen chains of an output meet in the tree.
//
// Wave w of a block runs the chains w, w + 8, w + 4, w + 12 of the block's
// tile one after the other: (l_w + l_w+8) + (l_w+4 + l_w+12) is its share
// of the tree, and the shares of the four waves meet in LDS as (W0 + W2) +
// (W1 + W3). The waves share no operands, so the loop has no LDS and no
// barriers: the input rows come from a copy laid out as the MFMA operand
// (chain_tile_kernel: 16 bytes a lane give four MFMA steps), the weights
// from the layer's lane-chain layout (four consecutive steps a lane,
// widened, then a 4 x 4 transpose between registers and the wave's
// quarters), the next 16 steps' loads in flight while 16 run.
//
// Bound: the f32 matrix rate (139 TFLOP/s in a register-only loop). In
// launches of 8 rows Whisper base's encoder products (1500 rows, 512 x 512
// to 2048 x 512, and the stem) were bound by the launches and the vector
// chains: 23.5 ms for its stem and two layers; here 0.47 ms, 0.07 ms of it
// the operand copies.
#include "float_weights.h"

#include <type_traits>

namespace trit {
namespace {

typedef float f32x4 __attribute__((ext_vector_type(4)));

constexpr int THREADS = 256;
constexpr int TILE = 16;         // MFMA rows and columns
constexpr int SB = 16;           // chain steps a 16-byte operand load covers
constexpr int KB = 16 * SB;      // inputs of a row in one block of the operand copy

int blocks_of_k(int k) { return (k + KB - 1) / KB; }
int row_tiles(int m) { return (m + TILE - 1) / TILE; }

// x (m x k) as operand blocks: block (chain i, step block b, row tile t) is
// 64 lanes x 4 floats, lane (row r, quarter q) holding steps 16 b + 4 j + q
// (j = 0..3) of row 16 t + r. Zero past m and k.
__global__ __launch_bounds__(THREADS) void chain_tile_kernel(const float* __restrict__ x, int m, int k, int tiles,
                                                             float4* __restrict__ out) {
    constexpr int PITCH = KB + 1;
    __shared__ float t[TILE * PITCH];
    const int rt = blockIdx.x, b = blockIdx.y, nb = gridDim.y;
    const int tid = threadIdx.x;
    // A row's 256 inputs by consecutive threads.
#pragma unroll
    for (int r = 0; r < TILE; ++r) {
        const int row = rt * TILE + r, col = b * KB + tid;
        t[r * PITCH + tid] = row < m && col < k ? x[(size_t)row * k + col] : 0.0f;
    }
    __syncthreads();
    const int lane = tid % WAVE, r = lane % 16, q = lane / 16;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const int i = tid / WAVE + 4 * j;
        const float* p = t + r * PITCH + 16 * q + i;
        out[(((size_t)i * nb + b) * tiles + rt) * WAVE + lane] = make_float4(p[0], p[64], p[128], p[192]);
    }
}

// Four consecutive chain steps of one weight row as loaded.
template <int K>
struct Raw;
template <>
struct Raw<WK_F16> { uint2 v; };
template <>
struct Raw<WK_F32> { float4 v; };
template <>
struct Raw<WK_Q8> { uint32_t v; float2 s; };

// Steps s0..s0+3 of the chain at `c`; the steps from s_count on are -0
// (times the copy's +0 that is -0, which leaves any accumulator as it is).
// VEC: s_count is a multiple of 4, so the four are all in or all out and
// load in one piece; else one element at a time.
template <int K, bool VEC>
__device__ __forceinline__ Raw<K> load_steps(const typename WT<K>::E* c, const float* row_scales, int s0,
                                             int s_count) {
    Raw<K> r;
    if constexpr (K == WK_F16) {
        if constexpr (VEC) {
            r.v = s0 < s_count ? *(const uint2*)(c + s0) : make_uint2(0x80008000u, 0x80008000u);
        } else {
            uint32_t h[4];
#pragma unroll
            for (int j = 0; j < 4; ++j) h[j] = s0 + j < s_count ? c[s0 + j] : 0x8000u;
            r.v = make_uint2(h[0] | h[1] << 16, h[2] | h[3] << 16);
        }
    } else if constexpr (K == WK_F32) {
        if constexpr (VEC) {
            r.v = s0 < s_count ? *(const float4*)(c + s0) : make_float4(-0.0f, -0.0f, -0.0f, -0.0f);
        } else {
            float f[4];
#pragma unroll
            for (int j = 0; j < 4; ++j) f[j] = s0 + j < s_count ? c[s0 + j] : -0.0f;
            r.v = make_float4(f[0], f[1], f[2], f[3]);
        }
    } else {
        // Past the chain: code 0 times -0... as code 1 times scale -0.
        if constexpr (VEC) {
            const bool in = s0 < s_count;
            r.v = in ? *(const uint32_t*)(c + s0) : 0x01010101u;
            r.s = in ? *(const float2*)(row_scales + s0 / 2) : make_float2(-0.0f, -0.0f);
        } else {
            // s_count is even (k a multiple of 32): a scale's two steps are both in or both out.
            uint32_t v = 0;
            float s[2];
#pragma unroll
            for (int j = 0; j < 4; ++j) v |= (uint32_t)(uint8_t)(s0 + j < s_count ? c[s0 + j] : (int8_t)1) << (8 * j);
#pragma unroll
            for (int j = 0; j < 2; ++j) s[j] = s0 + 2 * j < s_count ? row_scales[s0 / 2 + j] : -0.0f;
            r.v = v;
            r.s = make_float2(s[0], s[1]);
        }
    }
    return r;
}

template <int K>
__device__ __forceinline__ void widen(const Raw<K>& r, float (&f)[4]) {
    if constexpr (K == WK_F16) {
        f[0] = f16_to_f32((uint16_t)(r.v.x & 0xffff));
        f[1] = f16_to_f32((uint16_t)(r.v.x >> 16));
        f[2] = f16_to_f32((uint16_t)(r.v.y & 0xffff));
        f[3] = f16_to_f32((uint16_t)(r.v.y >> 16));
    } else if constexpr (K == WK_F32) {
        f[0] = r.v.x;
        f[1] = r.v.y;
        f[2] = r.v.z;
        f[3] = r.v.w;
    } else {
#pragma unroll
        for (int j = 0; j < 4; ++j)
            f[j] = (float)(int8_t)(uint8_t)(r.v >> (8 * j)) * (j < 2 ? r.s.x : r.s.y);
    }
}

// Output tile: TM x TN tiles of 16 x 16 a block.
template <int K, bool VEC, int TM, int TN, bool GELU>
__global__ __launch_bounds__(THREADS, 2) void float_mfma_kernel(const float4* __restrict__ xt, int tiles, int nb,
                                                                const typename WT<K>::E* __restrict__ w,
                                                                const float* __restrict__ scales,
                                                                const float* __restrict__ bias, int n, int k,
                                                                int nbn, int nbm, GemvArgs a) {
    constexpr int BM = TM * TILE, BN = TN * TILE;
    __shared__ __align__(16) float part[4][BM * BN];
    if (a.skip && *a.skip) return;
    // Block b runs on XCD b % 8: the blocks of one XCD share weight columns.
    const int blk = blockIdx.x;
    int bn, bm;
    if (nbn % 8 == 0) {
        const int q = blk / 8;
        bn = blk % 8 + 8 * (q / nbm);
        bm = q % nbm;
    } else {
        bn = blk % nbn;
        bm = blk / nbn;
    }
    const int lane = threadIdx.x % WAVE, wave = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE);
    const int lr = lane % 16, q = lane / 16;
    const int s_count = chain_steps(k);
    const typename WT<K>::E* wrow[TN];
    const float* srow[TN];
#pragma unroll
    for (int j = 0; j < TN; ++j) {
        const int col = min(bn * BN + j * TILE + lr, n - 1);  // columns past n are not stored
        wrow[j] = w + (size_t)col * 16 * s_count;
        srow[j] = K == WK_Q8 ? scales + (size_t)col * (k / 32) : nullptr;
    }
    int rt[TM];
#pragma unroll
    for (int i = 0; i < TM; ++i) rt[i] = min(bm * TM + i, tiles - 1);

    float4 na[TM];
    Raw<K> nw[TN];
    auto chain_of = [&](int c) { return wave + (c & 1) * 8 + (c >> 1) * 4; };  // w, w + 8, w + 4, w + 12
    auto fetch = [&](int c, int b) {
        const int i = chain_of(c);
#pragma unroll
        for (int t = 0; t < TM; ++t) na[t] = xt[(((size_t)i * nb + b) * tiles + rt[t]) * WAVE + lane];
#pragma unroll
        for (int j = 0; j < TN; ++j)
            nw[j] = load_steps<K, VEC>(wrow[j] + (size_t)i * s_count, srow[j], SB * b + 4 * q, s_count);
    };
    f32x4 sum[TM][TN], pair[TM][TN];
    fetch(0, 0);
#pragma unroll
    for (int c = 0; c < 4; ++c) {
        f32x4 acc[TM][TN];
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j) acc[i][j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll 1
        for (int b = 0; b < nb; ++b) {
            float xa[TM][4], wb[TN][4];
#pragma unroll
            for (int i = 0; i < TM; ++i) {
                xa[i][0] = na[i].x;
                xa[i][1] = na[i].y;
                xa[i][2] = na[i].z;
                xa[i][3] = na[i].w;
            }
#pragma unroll
            for (int j = 0; j < TN; ++j) {
                widen<K>(nw[j], wb[j]);
                transpose_quarters(wb[j]);
            }
            if (b + 1 < nb) fetch(c, b + 1);
            else if (c < 3) fetch(c + 1, 0);
#pragma unroll
            for (int t = 0; t < 4; ++t)
#pragma unroll
                for (int i = 0; i < TM; ++i)
#pragma unroll
                    for (int j = 0; j < TN; ++j)
                        acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(xa[i][t], wb[j][t], acc[i][j], 0, 0, 0);
        }
        // The tree: l_w + l_w+8, then that plus l_w+4 + l_w+12.
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j) {
                if (c == 0) sum[i][j] = acc[i][j];
                if (c == 1) sum[i][j] = sum[i][j] + acc[i][j];
                if (c == 2) pair[i][j] = acc[i][j];
                if (c == 3) sum[i][j] = sum[i][j] + (pair[i][j] + acc[i][j]);
            }
    }
    // Register r of a lane is output (row 4 q + r, column lr) of a tile.
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
            for (int r = 0; r < 4; ++r) part[wave][(i * TILE + 4 * q + r) * BN + j * TILE + lr] = sum[i][j][r];
    __syncthreads();
    for (int e = threadIdx.x; e < BM * BN; e += THREADS) {
        const int row = bm * BM + e / BN, col = bn * BN + e % BN;
        if (row >= a.m || col >= n) continue;
        float v[1] = {(part[0][e] + part[2][e]) + (part[1][e] + part[3][e])};
        finish_outputs<GELU>(v, bias, {col}, a.relu);
        const size_t at = (size_t)row * n + col;
        a.y[at] = a.epilogue == EPI_RESIDUAL ? a.residual[at] + v[0] : v[0];
    }
}

// Tiles of 32 rows x 64 columns from 512 blocks of them, else 32 x 16: between
// one block a CU and two, half the CUs would wait for the others' second. (A
// whole round of long f16 or Q8 rows takes them too.) 16 columns against 64, us, by
// the blocks of 64: f16 512x512 192 13.2, 14.7, 320 17.7, 21.9, 376 21.6, 23.8, 512
// 27.0, 26.0, 1024 46.8, 38.9; 512x2048 256 37.6, 35.7, 376 52.7, 59.1, 512 81.8,
// 60.8; f32 512x2048 256 38.8, 42.3, 376 53.6, 62.6, 512 82.3, 64.7.
template <int K, bool VEC>
void launch_tiles(const Layer& L, const GemvArgs& a, const float4* xt, hipStream_t s) {
    using E = typename WT<K>::E;
    const int tiles = row_tiles(a.m), nb = blocks_of_k(L.k), nbm = (a.m + 31) / 32;
    auto go = [&](auto TN_) {
        constexpr int TN = decltype(TN_)::value;
        const int nbn = (L.n + TN * TILE - 1) / (TN * TILE);
        hipLaunchKernelGGL((a.gelu ? float_mfma_kernel<K, VEC, 2, TN, true> : float_mfma_kernel<K, VEC, 2, TN, false>),
                           dim3(nbn * nbm), dim3(THREADS), 0, s, xt, tiles, nb, L.codes.as<E>(),
                           K == WK_Q8 ? L.scales.as<float>() : nullptr, L.bias.as<float>(), L.n, L.k, nbn, nbm, a);
    };
    const int64_t blocks = (int64_t)((L.n + 63) / 64) * nbm;
    const bool round = K != WK_F32 && L.k >= 1024 && blocks >= 224 && blocks <= 256;
    if (blocks >= 512 || round) go(std::integral_constant<int, 4>{});
    else go(std::integral_constant<int, 1>{});
}

template <int K>
void launch_kind(const Layer& L, const GemvArgs& a, const float4* xt, hipStream_t s) {
    if (chain_steps(L.k) % 4 == 0) launch_tiles<K, true>(L, a, xt, s);
    else launch_tiles<K, false>(L, a, xt, s);
}

}  // namespace

namespace {

// Whether 9 to 16 rows are shorter as two launches of up to 8 (gemv_float's
// chunked kernel, which stages aligned rows of whole 16-byte weight steps): a
// layer of few outputs fills those with one pass over its weights, while here
// the operand copy, and for Q8 the widening in every row tile, come on top.
// Rows 9 and 16, two launches against this file's kernels: f16 512x512 7.0 and
// 7.6 us against 8.3 and 8.8, 512x8192 38 and 49 against 48 and 48, 1024x4096 25
// and 33 against 27 and 27, 2048x4096 42 and 59 against 29 and 31; Q8 512x1024
// 9.0 and 10.5 against 12.6 and 13.1, 2048x1024 13.3 and 18.7 against 12.5 and
// 13.1; f32 256x2048 16.7 and 19.3 against 17.9 and 18.2. f16 rows of 1024 and
// 2048 have a kernel of their own there that is slower (14.6 and 21.1 against
// 11.8 and 12.3).
bool few_rows_by_eights(const Layer& L, const GemvArgs& a) {
    if (a.m > 16 || a.gelu || ((uintptr_t)a.x & 15) != 0) return false;
    const bool most = a.m <= 12;
    switch (L.kind) {
        case F16: return L.k % 128 == 0 && L.k != 1024 && L.k != 2048 && L.k >= 512 && L.n <= (most ? 1024 : 512);
        case F32: return L.k % 64 == 0 && L.k >= 1024 && L.k <= 2048 && L.n <= 512 && most;
        default: return L.k % 256 == 0 && L.k >= 512 && L.n <= (most || L.k <= 2048 ? 1024 : 512);
    }
}

}  // namespace

bool gemm_float_mfma_supported(const Layer& L, const GemvArgs& a) {
    return float_kind(L.kind) && a.m >= 9 && !a.norm_w && a.epilogue != EPI_SILU_PAIR && !few_rows_by_eights(L, a);
}

size_t gemm_float_scratch_bytes(int m, int k) {
    return (size_t)row_tiles(m) * TILE * blocks_of_k(k) * KB * sizeof(float);
}

void gemm_float_mfma(const Layer& L, GemvArgs a, void* scratch, size_t scratch_bytes, hipStream_t s) {
    if (!gemm_float_mfma_supported(L, a)) fail("float rows: not a product the f32 matrix cores take");
    const size_t per_tile = gemm_float_scratch_bytes(1, L.k);
    const size_t fit = scratch_bytes / per_tile * TILE;  // rows a pass
    if (fit == 0) fail("float rows: the scratch does not hold 16 rows");
    const int m = a.m, rows = (int)(fit < (size_t)m ? fit : (size_t)m);
    const float* x = a.x;
    float* y = a.y;
    const float* residual = a.residual;
    for (int r0 = 0; r0 < m; r0 += rows) {
        a.m = m - r0 < rows ? m - r0 : rows;
        a.x = x + (size_t)r0 * L.k;
        a.y = y + (size_t)r0 * L.n;
        if (residual) a.residual = residual + (size_t)r0 * L.n;
        hipLaunchKernelGGL(chain_tile_kernel, dim3(row_tiles(a.m), blocks_of_k(L.k)), dim3(THREADS), 0, s, a.x, a.m,
                           L.k, row_tiles(a.m), (float4*)scratch);
        TRIT_HIP(hipGetLastError());
        const float4* xt = (const float4*)scratch;
        switch (L.kind) {
            case F16: launch_kind<WK_F16>(L, a, xt, s); break;
            case F32: launch_kind<WK_F32>(L, a, xt, s); break;
            default: launch_kind<WK_Q8>(L, a, xt, s); break;
        }
        TRIT_HIP(hipGetLastError());
    }
}

}  // namespace trit
