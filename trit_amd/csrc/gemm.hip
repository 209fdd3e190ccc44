// Integer products of many rows (prompt prefill) on the matrix cores:
// Q8_0 (and Q4_K requantized to it) with 32-value groups, Trit int8 and
// ternary with 128-value groups.
//
// The values are Trit's, bit for bit, as in the small-batch kernels
// (src/cpu/int8.rs:525-584, src/cpu/v2/product.rs:389-423):
//   y[f][r] = chain over groups g in order of
//             total = fma(f32(dot_g), ws[r][g] * xs[f][g], total), from +0,
// where dot_g is the exact i32 dot of the group's weight codes and the
// activation codes of Trit's quantizer (src/cpu/kernels.rs:661-807). The
// matrix cores make the i32 group dots (v_mfma_i32_32x32x32_i8: one 32-wide
// step is one Q8_0 group, four steps one int8 group); the f32 chain runs on
// the vector ALUs in group order, per output, in the MFMA's own register
// layout.
//
// Passes:
//  1. (RMSNorm rows) row_norm_kernel: each row's factor, with the same sum
//     tree as the small-batch kernel's prologue;
//  2. quantize_kernel: Trit's activation quantizer over all rows into codes
//     (m x k) and group scales stored group-major (g x mpad), so that a
//     lane's four consecutive output rows read one 16-byte load;
//  3. the product: gemm_dma_kernel where k is a multiple of 128,
//     gemm_ternary_kernel for ternary layers, else gemm_wide_kernel (large
//     products) or gemm_kernel: 256 threads = 2 x 2 waves over 64 rows of x
//     and 128 weight rows. K runs in 256-byte chunks staged through LDS (the
//     last one zero past k): 16 threads read a row's 256 contiguous bytes,
//     and the next chunk's loads are in flight while this one computes. A
//     wave owns 32 rows of x by two 32-row MFMA tiles of weights (or, for
//     the SwiGLU pair, the gate tile and its up tile), so every (row,
//     output) total stays in one lane's registers from the first group to
//     the epilogue.
#include "gemm_kernels.h"

namespace trit {
namespace {

int round_up(int v, int to) { return (v + to - 1) / to * to; }

// RMSNorm factor per row: each 256-value chunk's squares summed by a
// shuffle butterfly over one wave, the chunks added in order from lane 0 --
// the bits of the small-batch kernel's prologue (gemv.hip), so a prompt row
// gets the same factor on either path. One wave per row, k % 256 == 0.
__global__ __launch_bounds__(WAVE) void row_norm_kernel(const float* __restrict__ x, int k, float eps,
                                                         float* __restrict__ inv, const int* skip) {
    if (skip && *skip) return;
    const int row = blockIdx.x, lane = threadIdx.x;
    float sum = 0.0f;
    for (int c = 0; c < k / 256; ++c) {
        const float4 v = *(const float4*)(x + (size_t)row * k + c * 256 + lane * 4);
        float part = (v.x * v.x + v.y * v.y) + (v.z * v.z + v.w * v.w);
#pragma unroll
        for (int off = WAVE / 2; off > 0; off >>= 1) part += __shfl_xor(part, off);
        sum += __shfl(part, 0);
    }
    if (lane == 0) inv[row] = 1.0f / __builtin_sqrtf(sum / (float)k + eps);
}

// Byte of activation code (row, col) in the ternary product's operand order:
// blocks of 32 rows by one 128-group, in a block the four MFMA steps of 64
// lanes x 16 codes (step s, lane (row, half h): columns 64 h + 16 s ..), so a
// wave's operand load is 1 KB in one piece.
__device__ __forceinline__ size_t ternary_code(int row, int col, int k) {
    const int g = col / 128, h = col / 64 % 2, s = col / 16 % 4;
    return (((size_t)(row / 32) * (k / 128) + g) * 4 + s) * 1024 + (h * 32 + row % 32) * 16 + col % 16;
}

// Trit's activation quantizer (src/cpu/kernels.rs:661-737), G/4 threads per
// group, four values a thread; rows [m, mpad) get zero scales. TERN: codes in
// the ternary product's order, else row-major.
template <int G, bool HALF, bool TERN = false>
__global__ __launch_bounds__(256) void quantize_kernel(const float* __restrict__ x, int m, int mpad, int k,
                                                       const float* __restrict__ norm_w,
                                                       const float* __restrict__ inv, int8_t* __restrict__ xq,
                                                       float* __restrict__ xs, const int* skip) {
    if (skip && *skip) return;
    constexpr int TPG = G / 4;
    const int ipr = k / 4;  // items per row
    const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
    const bool live = i < (size_t)mpad * ipr;
    const int row = live ? (int)(i / ipr) : 0;
    const int col = live ? (int)(i - (size_t)row * ipr) * 4 : 0;
    const bool real = live && row < m;
    float4 v = real ? *(const float4*)(x + (size_t)row * k + col) : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    if (norm_w && real) {
        const float f = inv[row];
        const float4 w = *(const float4*)(norm_w + col);
        v.x = v.x * (f * w.x);
        v.y = v.y * (f * w.y);
        v.z = v.z * (f * w.z);
        v.w = v.w * (f * w.w);
    }
    float peak = __builtin_fmaxf(__builtin_fmaxf(__builtin_fabsf(v.x), __builtin_fabsf(v.y)),
                                 __builtin_fmaxf(__builtin_fabsf(v.z), __builtin_fabsf(v.w)));
#pragma unroll
    for (int off = TPG / 2; off > 0; off >>= 1) peak = __builtin_fmaxf(peak, __shfl_xor(peak, off));
    const float scale = peak > 0.0f ? peak / 127.0f : 1.0f;
    const float q = 1.0f / scale;
    const int c0 = act_code(v.x * q), c1 = act_code(v.y * q);
    const int c2 = act_code(v.z * q), c3 = act_code(v.w * q);
    if (real) *(uint32_t*)(xq + (TERN ? ternary_code(row, col, k) : (size_t)row * k + col)) = pack4(c0, c1, c2, c3);
    if (live && col % G == 0) xs[(size_t)(col / G) * mpad + row] = real ? (HALF ? f16_round(scale) : scale) : 0.0f;
}

// The same over the im2col rows of a kernel-3, stride-2, padding-1 2-D
// convolution, from its [map][bin][time][channel] input: column c * 9 + tap of
// a row is tap's pixel's channel c, zero outside the map
// (src/models/families/qwen3_asr.rs:408-428). A row's nine pixels go to LDS
// (each a run of channels; the pitch of 15 mod 32 floats spreads the taps over
// the banks), the groups are read from there in column order, so the columns
// never reach memory in f32: with them written and read back, the 24000 rows
// of 4320 columns that 30 s of audio make took 250 us + 150 us. An XCD takes
// consecutive rows, which share pixels.
constexpr int CONV_ROWS = 4;  // rows a block

__host__ __device__ constexpr int conv_pitch(int channels) { return (channels + 16) / 32 * 32 + 15; }

template <int G, bool HALF>
__global__ __launch_bounds__(256) void quantize_conv_kernel(ConvInput in, int m, int mpad, int8_t* __restrict__ xq,
                                                            float* __restrict__ xs, const int* skip) {
    if (skip && *skip) return;
    extern __shared__ float px[];  // [tap][pitch]
    constexpr int TPG = G / 4;
    const int ch = in.channels, pitch = conv_pitch(ch), k = 9 * ch;
    const int ob = (in.bins + 1) / 2, ot = (in.times + 1) / 2;
    const int id = (int)(blockIdx.x % 8) * (int)(gridDim.x / 8) + (int)(blockIdx.x / 8);
    for (int row = id * CONV_ROWS; row < min((id + 1) * CONV_ROWS, mpad); ++row) {
        if (row >= m) {
            for (int g = threadIdx.x; g < k / G; g += 256) xs[(size_t)g * mpad + row] = 0.0f;
            continue;
        }
        const int xo = row % ot, yo = row / ot % ob, map = row / (ot * ob);
        __syncthreads();  // the row before is read
        for (int i = threadIdx.x; i < 9 * (ch / 4); i += 256) {
            const int tap = i / (ch / 4), c = (i - tap * (ch / 4)) * 4;
            const int sy = 2 * yo + tap / 3 - 1, sx = 2 * xo + tap % 3 - 1;
            float4 v = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
            if (sy >= 0 && sy < in.bins && sx >= 0 && sx < in.times)
                v = *(const float4*)(in.in + (((size_t)map * in.bins + sy) * in.times + sx) * ch + c);
            float* to = px + tap * pitch + c;
            to[0] = v.x;
            to[1] = v.y;
            to[2] = v.z;
            to[3] = v.w;
        }
        __syncthreads();
        // k / 4 is a multiple of TPG, so a group's lanes take an item together.
        for (int i = threadIdx.x; i < k / 4; i += 256) {
            float v[4];
            int c = 4 * i / 9, tap = 4 * i - 9 * c;
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                v[u] = px[tap * pitch + c];
                if (++tap == 9) {
                    tap = 0;
                    ++c;
                }
            }
            float peak = __builtin_fmaxf(__builtin_fmaxf(__builtin_fabsf(v[0]), __builtin_fabsf(v[1])),
                                         __builtin_fmaxf(__builtin_fabsf(v[2]), __builtin_fabsf(v[3])));
#pragma unroll
            for (int off = TPG / 2; off > 0; off >>= 1) peak = __builtin_fmaxf(peak, __shfl_xor(peak, off));
            const float scale = peak > 0.0f ? peak / 127.0f : 1.0f;
            const float q = 1.0f / scale;
            *(uint32_t*)(xq + (size_t)row * k + 4 * i) =
                pack4(act_code(v[0] * q), act_code(v[1] * q), act_code(v[2] * q), act_code(v[3] * q));
            if (4 * i % G == 0) xs[(size_t)(4 * i / G) * mpad + row] = HALF ? f16_round(scale) : scale;
        }
    }
}

int group_of(const Layer& L) { return L.kind == INT8 || L.kind == TERNARY ? 128 : 32; }

// Rows of x codes a product's scratch holds: whole 32-row operand blocks for a
// ternary layer (64 with the scales' padding).
int code_rows(const Layer& L, int m) { return L.kind == TERNARY ? round_up(m, BM) : m; }

GemmScratch carve(void* base, const Layer& L, int m) {
    const int mpad = round_up(m, BM), k = L.k;
    auto al = [](size_t v) { return (v + 255) & ~(size_t)255; };
    char* p = (char*)base;
    GemmScratch s;
    s.mpad = mpad;
    s.xq = (int8_t*)p;
    p += al((size_t)code_rows(L, m) * k);
    s.xs = (float*)p;
    p += al((size_t)(k / 32) * mpad * 4);
    s.inv = (float*)p;
    return s;
}

}  // namespace

bool gemm_supported(const Layer& L, const GemvArgs& a) {
    if (L.kind != Q8_0 && L.kind != Q4_K && L.kind != INT8 && L.kind != TERNARY) return false;
    if (L.kind == TERNARY && a.epilogue == EPI_SILU_PAIR) return false;
    // k a multiple of the group (a partial last chunk of K is zero past k);
    // RMSNorm computed here takes whole 256-value chunks.
    if (L.k % group_of(L) != 0) return false;
    if (a.epilogue == EPI_SILU_PAIR && (L.n / 2) % 64 != 0) return false;
    if (a.norm_w && !a.norm_inv && L.k % KC != 0) return false;
    // 32-bit byte offsets into the codes of x and of the weights.
    if ((int64_t)a.m * L.k >= (int64_t)1 << 31 || (int64_t)L.n * L.k >= (int64_t)1 << 32) return false;
    return a.m >= 1;
}

bool ternary_by_eights(const Layer& L, const GemvArgs& a) {
    if (L.kind != TERNARY || a.gelu || a.m < 9 || a.m > 16 || L.n % 4 != 0 || L.k > 6784) return false;
    if (a.m == 9) return L.k >= 3584 && L.n <= 2048;
    return L.n <= 1024 && L.k >= (a.m == 10 ? 4096 : a.m <= 12 ? 5120 : 6144);
}

size_t gemm_scratch_bytes(int m, int k) {
    const size_t mpad = (size_t)round_up(m, BM);
    auto al = [](size_t v) { return (v + 255) & ~(size_t)255; };
    return al((size_t)m * k) + al((size_t)(k / 32) * mpad * 4) + al(mpad * 4);
}

size_t gemm_scratch_bytes(const Layer& L, int m) { return gemm_scratch_bytes(code_rows(L, m), L.k); }

bool gemm_conv_supported(const Layer& L, const ConvInput& in) {
    return !float_kind(L.kind) && L.kind != TERNARY && L.k == 9 * in.channels && in.channels % 4 == 0 &&
           (size_t)9 * conv_pitch(in.channels) * 4 <= 64 * 1024;
}

void gemm_int(const Layer& L, const GemvArgs& a, void* scratch, hipStream_t s, const ConvInput* conv) {
    if (!gemm_supported(L, a)) fail("gemm: layer " + std::to_string(L.n) + "x" + std::to_string(L.k) +
                                    " is not a shape the matrix-core product takes");
    const GemmScratch sc = carve(scratch, L, a.m);
    const float* inv = a.norm_inv;
    if (a.norm_w && !inv) {
        hipLaunchKernelGGL(row_norm_kernel, dim3(a.m), dim3(WAVE), 0, s, a.x, L.k, a.eps, sc.inv, a.skip);
        TRIT_HIP(hipGetLastError());
        inv = sc.inv;
    }
    const int G = group_of(L);
    const size_t items = (size_t)sc.mpad * (L.k / 4);
    const int qblocks = (int)((items + 255) / 256);
    if (conv) {
        if (!gemm_conv_supported(L, *conv) || a.norm_w) fail("gemm: not a convolution the quantizer takes");
        const size_t lds = (size_t)9 * conv_pitch(conv->channels) * 4;
        const int blocks = (sc.mpad / CONV_ROWS + 7) / 8 * 8;
        if (G == 32)
            hipLaunchKernelGGL((quantize_conv_kernel<32, true>), dim3(blocks), dim3(256), lds, s, *conv, a.m, sc.mpad,
                               sc.xq, sc.xs, a.skip);
        else
            hipLaunchKernelGGL((quantize_conv_kernel<128, false>), dim3(blocks), dim3(256), lds, s, *conv, a.m,
                               sc.mpad, sc.xq, sc.xs, a.skip);
    } else if (L.kind == TERNARY)
        hipLaunchKernelGGL((quantize_kernel<128, false, true>), dim3(qblocks), dim3(256), 0, s, a.x, a.m, sc.mpad, L.k,
                           a.norm_w, inv, sc.xq, sc.xs, a.skip);
    else if (G == 32)
        hipLaunchKernelGGL((quantize_kernel<32, true>), dim3(qblocks), dim3(256), 0, s, a.x, a.m, sc.mpad, L.k,
                           a.norm_w, inv, sc.xq, sc.xs, a.skip);
    else
        hipLaunchKernelGGL((quantize_kernel<128, false>), dim3(qblocks), dim3(256), 0, s, a.x, a.m, sc.mpad, L.k,
                           a.norm_w, inv, sc.xq, sc.xs, a.skip);
    TRIT_HIP(hipGetLastError());
    if (a.gelu && a.epilogue != EPI_SILU_PAIR) return gemm_gelu(L, a, sc, s);
    return launch_product<false>(L, a, sc, s);
}

}  // namespace trit
