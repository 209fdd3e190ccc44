// Trit's attention of many query rows on the f32 matrix cores, bit for bit
// the vector kernels' results (attention_kernel, attention_rows_kernel in
// decoder.hip; src/layers.rs:442-504,571-587): scores are fused chains over
// the dims from +0, the softmax sum runs over the keys in order, outputs are
// fused chains over the keys from +0. v_mfma_f32_16x16x4_f32 is such a
// chain: four fused multiply-adds in k order onto each accumulator, every
// one rounded to nearest even, subnormals kept.
//
// A block takes 16 query rows of one head, its W waves every W-th tile of
// 16 keys:
//  1. S^T = K Q^T a tile at a time, q (times 1 / sqrt(hd)) in registers as
//     the MFMA operand, a key's dims loaded four a lane and transposed
//     between registers and quarters. The scores of every key stay in
//     registers (NT tiles a wave: 16 rows x 1564 keys are 100 KB, which in
//     LDS would leave one block a CU);
//  2. the rows' maxima over lanes and waves, the exponentials in place;
//  3. the sums, in key order: the exponentials pass through LDS in chunks of
//     4 W tiles (two buffers), wave 0 adding one chunk while the waves write
//     the next;
//  4. O^T = V^T P^T: the probabilities, transposed to the MFMA operand, pass
//     through the same buffers; wave w chains the dims of its VE 16-dim
//     tiles over every key, the values loaded four tiles ahead.
// Blocks go to the XCDs head by head (block b runs on XCD b % 8), so an
// XCD's L2 holds the keys and values of the heads it works on; within a head
// the last rows first (a causal prompt's longest).
//
// Bound: the f32 matrix rate (139 TFLOP/s in a register-only loop) and, one
// block a CU, the serial sum of phase 3 (about 10 cycles a key); 2-3 blocks a
// CU overlap each other's phases. Vector instructions share the SIMDs with the
// MFMAs, so addresses are 32-bit offsets and only tiles at an edge are masked
// (with 64-bit row addresses and a mask a value, 278 us and 210 us below).
// Whisper large-v3's layer (1500 rows, 20 heads of 64, 11.5 GFLOP): 232 us
// against 782 us for the vector kernel's 4 rows a block; a causal prompt of 1564
// rows (16 heads of 128, 10 GFLOP of visible keys): 186 us against 494 us.
#pragma once

#include <cmath>

#include "decoder_impl.h"
#include "device.h"
#include "internal.h"

namespace trit {
namespace {

typedef float f32x4 __attribute__((ext_vector_type(4)));

constexpr int TILE = 16;

// Four consecutive elements of a key, or VE of a value, as loaded.
template <typename KV>
struct Four;
template <>
struct Four<float> { float4 v; };
template <>
struct Four<_Float16> { uint2 v; };

__device__ __forceinline__ void load4(const float* p, Four<float>& r) { r.v = *(const float4*)p; }
__device__ __forceinline__ void load4(const _Float16* p, Four<_Float16>& r) { r.v = *(const uint2*)p; }
__device__ __forceinline__ void widen4(const Four<float>& r, float (&f)[4]) {
    f[0] = r.v.x;
    f[1] = r.v.y;
    f[2] = r.v.z;
    f[3] = r.v.w;
}
__device__ __forceinline__ void widen4(const Four<_Float16>& r, float (&f)[4]) {
    f[0] = f16_to_f32((uint16_t)(r.v.x & 0xffff));
    f[1] = f16_to_f32((uint16_t)(r.v.x >> 16));
    f[2] = f16_to_f32((uint16_t)(r.v.y & 0xffff));
    f[3] = f16_to_f32((uint16_t)(r.v.y >> 16));
}

template <typename KV, int VE>
struct alignas(sizeof(KV) * VE) Values {
    KV e[VE];
};

template <typename KV, int HD, int NT, int W>
__global__ __launch_bounds__(64 * W, W == 4 && (HD == 64 || sizeof(KV) == 2) ? 3 : 2) void attention_rows_mfma_kernel(RowsArgs a) {
    constexpr int VE = HD / TILE > W ? HD / TILE / W : 1;  // 16-dim output tiles a wave
    constexpr int PVW = HD / TILE / VE;                    // waves with output tiles
    constexpr int CT = 4 * W;                              // tiles a chunk
    constexpr int CHUNKS = (NT + 3) / 4;
    __shared__ __align__(16) float4 buf[2][CT * WAVE];
    __shared__ float red[W][TILE];
    __shared__ float inv_of[TILE];
    if (a.st->done) return;
    const int pos = a.st->pos;
    // Head-major block ids, an eighth of them on each XCD.
    const int per = gridDim.x / 8;
    const int id = (int)(blockIdx.x % 8) * per + (int)(blockIdx.x / 8);
    if (id >= a.heads * a.tiles) return;
    const int h = id / a.tiles, tile = a.tiles - 1 - id % a.tiles;
    const int g = h / (a.heads / a.kvh);
    // The tile's window (one window of all rows but for windowed encoders).
    const int win = tile / a.window_tiles, row0 = (tile - win * a.window_tiles) * TILE;
    const int first = win * a.window;                       // the window's first row
    const int rows = min(a.window, a.rows - first);
    const int nr = min(TILE, rows - row0);
    const int tk = pos + rows;
    // Causal rows see no key past kmax; those keys weigh exp_trit(-inf) /
    // sum, at most 1.2e-38: with f16 values (|v| <= 65504) such a term is
    // below 7.7e-34, under half a step of any |out| >= 2^-80, and the chains
    // stop at kmax (nearer 0 they go on, below); f32 values take every key.
    // (Sums of less than 1: the row's maximum is infinite or all its scores
    // are NaN, every key weighs the same, and sum and chains go on. An
    // infinite f16 value past kmax, which Trit's chain would carry into this
    // row, is left out here; the forward's last row sees it in both.)
    const int kmax = a.causal ? min(tk, pos + row0 + nr) : tk;
    const int kend = sizeof(KV) == 2 ? kmax : tk;
    const int ntiles = (kend + TILE - 1) / TILE;
    const int t = threadIdx.x;
    const int lane = t % WAVE, w = __builtin_amdgcn_readfirstlane(t / WAVE);
    const int lr = lane % 16, q = lane / 16;
    // Keys and values at 32-bit byte offsets from the head's first (the host
    // checks they fit).
    const char* K = (const char*)((const KV*)a.k + (size_t)g * a.head_stride + (size_t)first * a.pos_stride);
    const char* V = (const char*)((const KV*)a.v + (size_t)g * a.head_stride + (size_t)first * a.pos_stride);
    const uint32_t pitch = (uint32_t)(a.pos_stride * sizeof(KV));

    // 1. Scores. Operand register i of a lane: dim 4 i + q of query row lr
    // (rows past nr repeat the last one; nothing of them is stored).
    float qf[HD / 4];
    {
        const float scale = 1.0f / __builtin_sqrtf((float)HD);
        const float* qr = a.q + (size_t)(first + row0 + min(lr, nr - 1)) * a.q_stride + (size_t)h * HD + q;
#pragma unroll
        for (int i = 0; i < HD / 4; ++i) qf[i] = qr[4 * i] * scale;
    }
    const int visible = a.causal ? pos + row0 + lr + 1 : tk;       // of row lr
    const int all_visible = a.causal ? pos + row0 + 1 : tk;        // of every row
    float s[NT][4];  // s[j][r]: key 16 (w + W j) + 4 q + r of row lr
    float best = -INFINITY;
    Four<KV> next[HD / 16];
    const uint32_t key_off = (uint32_t)(TILE * w + lr) * pitch, last_off = (uint32_t)(kmax - 1) * pitch;
    auto fetch = [&](int j) {
        // (Past the last key: that key again; its scores are masked.)
        const uint32_t off = min(key_off + (uint32_t)(TILE * W * j) * pitch, last_off) + 4 * q * (uint32_t)sizeof(KV);
#pragma unroll
        for (int i = 0; i < HD / 16; ++i) load4((const KV*)(K + off) + 16 * i, next[i]);
    };
    fetch(0);
#pragma unroll
    for (int j = 0; j < NT; ++j) {
        const int key0 = TILE * (w + W * j);
        if (key0 < kmax) {
            Four<KV> cur[HD / 16];
#pragma unroll
            for (int i = 0; i < HD / 16; ++i) cur[i] = next[i];
            if (j + 1 < NT) fetch(j + 1);
            f32x4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
            for (int i = 0; i < HD / 16; ++i) {
                float f[4];
                widen4(cur[i], f);
                transpose_quarters(f);
#pragma unroll
                for (int u = 0; u < 4; ++u) acc = __builtin_amdgcn_mfma_f32_16x16x4f32(f[u], qf[4 * i + u], acc, 0, 0, 0);
            }
            if (key0 + TILE > all_visible) {
#pragma unroll
                for (int r = 0; r < 4; ++r) acc[r] = key0 + 4 * q + r < visible ? acc[r] : -INFINITY;
            }
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                s[j][r] = acc[r];
                best = __builtin_fmaxf(best, acc[r]);
            }
        } else {
#pragma unroll
            for (int r = 0; r < 4; ++r) s[j][r] = -INFINITY;
        }
    }

    // 2. Row lr's maximum.
    best = __builtin_fmaxf(best, __shfl_xor(best, 16));
    best = __builtin_fmaxf(best, __shfl_xor(best, 32));
    if (q == 0) red[w][lr] = best;
    __syncthreads();
    float mx = red[0][lr];
#pragma unroll
    for (int i = 1; i < W; ++i) mx = __builtin_fmaxf(mx, red[i][lr]);

    // 3. The exponentials, and the sums over the keys before kmax, in order.
    // Chunk c holds the tiles W (4 c) .. W (4 c + 4) - 1; in a tile, lane (row,
    // quarter) holds the keys 4 q .. 4 q + 3.
    float sum = 0.0f;
    auto add_chunk = [&](int c) {
        const int keys = min(TILE * CT, kmax - TILE * CT * c);  // may be none, when kmax < kend
        const float4* b = buf[c & 1] + lr;
        float4 cur[4], nxt[4];
        if (keys >= TILE) {
#pragma unroll
            for (int u = 0; u < 4; ++u) cur[u] = b[16 * u];
        }
        int i = 0;
        for (; TILE * (i + 1) <= keys; ++i) {
            const int o = (i + 1) % CT * WAVE;  // (past the keys: any tile, not added)
#pragma unroll
            for (int u = 0; u < 4; ++u) nxt[u] = b[o + 16 * u];
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                sum = sum + cur[u].x;
                sum = sum + cur[u].y;
                sum = sum + cur[u].z;
                sum = sum + cur[u].w;
            }
#pragma unroll
            for (int u = 0; u < 4; ++u) cur[u] = nxt[u];
        }
        for (int k = TILE * i; k < keys; ++k) sum = sum + ((const float*)(b + i * WAVE + k / 4 % 4 * 16))[k % 4];
    };
#pragma unroll
    for (int c = 0; c < CHUNKS; ++c) {
        if (CT * c < ntiles) {
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                const int j = 4 * c + u;
                if (j < NT) {
#pragma unroll
                    for (int r = 0; r < 4; ++r) s[j][r] = s[j][r] - mx;
                    exp_trit_n<true>(s[j]);
                    buf[c & 1][(u * W + w) * WAVE + lane] = make_float4(s[j][0], s[j][1], s[j][2], s[j][3]);
                }
            }
            __syncthreads();  // the chunk is written; the one before it is added up
            if (w == 0) add_chunk(c);
        }
    }
    if (t < TILE) {
        if (sum < 1.0f)
            for (int key = kmax; key < tk; ++key) sum = sum + exp_trit(-INFINITY);
        inv_of[t] = 1.0f / sum;
    }
    __syncthreads();
    const float inv = inv_of[lr];

    // 4. Outputs: register i of the operand is key 4 i + q of the tile. The
    // values past kend are -0: with any finite weight that leaves every chain
    // as it is.
    f32x4 out[VE];
#pragma unroll
    for (int u = 0; u < VE; ++u) out[u] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    const bool chains = w < PVW;
    const uint32_t dim_off = (uint32_t)(VE * (TILE * (chains ? w : 0) + lr)) * (uint32_t)sizeof(KV);
    const uint32_t lane_off = (uint32_t)q * pitch + dim_off;
    // Groups of four tiles, all but the last of whole tiles; nv: a group's values.
    const int whole = kend / (4 * TILE);
    Values<KV, VE> nv[16];
    auto fetch_value = [&](int group, int i) {
        const uint32_t at = (uint32_t)(4 * (16 * group + i)) * pitch;
        nv[i] = *(const Values<KV, VE>*)(V + at + lane_off);
    };
    auto fetch_last = [&](int group) {
        const uint32_t end = (uint32_t)(kend - 1) * pitch;
#pragma unroll
        for (int i = 0; i < 16; ++i)
            nv[i] = *(const Values<KV, VE>*)(V + min((uint32_t)(4 * (16 * group + i) + q) * pitch, end) + dim_off);
    };
    if (chains) {
        if (whole > 0) {
#pragma unroll
            for (int i = 0; i < 16; ++i) fetch_value(0, i);
        } else {
            fetch_last(0);
        }
    }
#pragma unroll
    for (int c = 0; c < CHUNKS; ++c) {
        if (CT * c < ntiles) {
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                const int j = 4 * c + u;
                if (j < NT) {
                    float p[4];
#pragma unroll
                    for (int r = 0; r < 4; ++r) p[r] = s[j][r] * inv;
                    transpose_quarters(p);
                    buf[c & 1][(u * W + w) * WAVE + lane] = make_float4(p[0], p[1], p[2], p[3]);
                }
            }
            __syncthreads();  // the chunk is written; the one before it is read
            if (chains) {
                const int n = min(CT, ntiles - CT * c);
#pragma unroll 1
                for (int i = 0; i < n; i += 4) {
                    const int group = CT / 4 * c + i / 4;
                    const float4* b = buf[c & 1] + i * WAVE + lane;
                    if (group < whole) {
                        const bool more = group + 1 < whole;
#pragma unroll
                        for (int u = 0; u < 4; ++u) {
                            const float4 p4 = b[u * WAVE];
                            const float p[4] = {p4.x, p4.y, p4.z, p4.w};
#pragma unroll
                            for (int x = 0; x < 4; ++x)
#pragma unroll
                                for (int v = 0; v < VE; ++v)
                                    out[v] = __builtin_amdgcn_mfma_f32_16x16x4f32((float)nv[4 * u + x].e[v], p[x], out[v],
                                                                                  0, 0, 0);
                            if (more) {
#pragma unroll
                                for (int x = 0; x < 4; ++x) fetch_value(group + 1, 4 * u + x);
                            }
                        }
                        if (!more && 4 * group + 4 < ntiles) fetch_last(group + 1);
                    } else {
#pragma unroll
                        for (int u = 0; u < 4; ++u) {
                            if (i + u >= n) break;
                            const float4 p4 = b[u * WAVE];
                            const float p[4] = {p4.x, p4.y, p4.z, p4.w};
#pragma unroll
                            for (int x = 0; x < 4; ++x)
#pragma unroll
                                for (int v = 0; v < VE; ++v) {
                                    const bool in = 4 * (16 * group + 4 * u + x) + q < kend;
                                    out[v] = __builtin_amdgcn_mfma_f32_16x16x4f32(in ? (float)nv[4 * u + x].e[v] : -0.0f,
                                                                                  p[x], out[v], 0, 0, 0);
                                }
                        }
                    }
                }
            }
        }
    }
    if (!chains || lr >= nr) return;
    // Register r of tile v: dim VE (16 w + 4 q + r) + v of row lr.
    float* o = a.out + (size_t)(first + row0 + lr) * a.heads * HD + (size_t)h * HD;
#pragma unroll
    for (int r = 0; r < 4; ++r)
#pragma unroll
        for (int v = 0; v < VE; ++v) {
            const int e = VE * (TILE * w + 4 * q + r) + v;
            float acc = out[v][r];
            if (kend < tk && (inv > 1.0f || !(__builtin_fabsf(acc) >= 0x1p-80f))) {
                const float pm = exp_trit(-INFINITY) * inv;
                for (int key = kend; key < tk; ++key)
                    acc = __builtin_fmaf(pm, (float)((const KV*)(V + (uint32_t)key * pitch))[e], acc);
            }
            o[e] = acc;
        }
}

template <typename KV, int HD, int NT, int W>
void launch(const RowsArgs& a, hipStream_t s) {
    const int blocks = (a.heads * a.tiles + 7) / 8 * 8;
    hipLaunchKernelGGL((attention_rows_mfma_kernel<KV, HD, NT, W>), dim3(blocks), dim3(64 * W), 0, s, a);
    TRIT_HIP(hipGetLastError());
}

// The smallest register budget that holds max_tk keys; false past 3200.
template <typename KV, int HD>
bool launch_budget(const RowsArgs& a, int max_tk, hipStream_t s) {
    if (max_tk <= 4 * 2 * TILE) launch<KV, HD, 2, 4>(a, s);
    else if (max_tk <= 4 * 8 * TILE) launch<KV, HD, 8, 4>(a, s);
    else if (max_tk <= 4 * 16 * TILE) launch<KV, HD, 16, 4>(a, s);
    else if (max_tk <= 4 * 25 * TILE) launch<KV, HD, 25, 4>(a, s);
    else if (max_tk <= 8 * 25 * TILE) launch<KV, HD, 25, 8>(a, s);
    else return false;
    return true;
}

}  // namespace
}  // namespace trit
