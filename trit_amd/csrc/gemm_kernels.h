// The many-row integer product kernels and their dispatch (gemm.hip, which
// says what they compute; gemm_gelu.hip).
#pragma once

#include "device.h"
#include "internal.h"

#include <type_traits>

namespace trit {

// The parts of a product's scratch.
struct GemmScratch {
    int8_t* xq;
    float* xs;
    float* inv;
    int mpad;
};

// The products with the GELU in their store: a code object of their own
// (gemm_gelu.hip), which a process that runs no encoder does not load.
void gemm_gelu(const Layer& L, const GemvArgs& a, const GemmScratch& sc, hipStream_t s);

namespace {

typedef int v4i __attribute__((ext_vector_type(4)));
typedef int v16i __attribute__((ext_vector_type(16)));

typedef float v16f __attribute__((ext_vector_type(16)));
typedef float v32f __attribute__((ext_vector_type(32)));

__device__ __forceinline__ v16f lower(const v32f& v) {
    return __builtin_shufflevector(v, v, 0, 1, 2, 3, 4, 5, 6, 7, 8, 9, 10, 11, 12, 13, 14, 15);
}
__device__ __forceinline__ v16f upper(const v32f& v) {
    return __builtin_shufflevector(v, v, 16, 17, 18, 19, 20, 21, 22, 23, 24, 25, 26, 27, 28, 29, 30, 31);
}

// Dots from the matrix cores as f32: accumulated on 0x4b400000, the bits of
// 1.5 * 2^23, a dot d is the bits of 1.5 * 2^23 + d exactly (|d| <= 128 * 128 *
// 127 < 2^22), so one subtraction gives f32(d) -- at nearly twice the rate of
// the conversion (16 of them 51 cycles a wave against 85, four waves a SIMD).
__device__ __forceinline__ v16i dot_base() {
    v16i m;
#pragma unroll
    for (int r = 0; r < 16; ++r) m[r] = 0x4b400000;
    // Sixteen registers, not a constant moved into every accumulator.
    asm("" : "+v"(m));
    return m;
}
__device__ __forceinline__ float dot_of(int bits) { return __builtin_bit_cast(float, bits) - 12582912.0f; }

constexpr int GEMM_THREADS = 256;
constexpr int BM = 64;  // rows of x per block: two waves of 32

constexpr int KC = 256;           // bytes of K per LDS chunk
constexpr int GPC = KC / 32;      // groups per chunk
constexpr int ROW_LDS = KC + 16;  // padded LDS row: rows 8 apart start 4 banks apart
constexpr int BN_ROWS = 128;      // weight rows per block

// One K chunk in LDS: the block's 64 x rows and 128 weight rows, and their
// group scales (weight scales widened to f32).
struct alignas(16) Stage {
    alignas(16) int8_t a[BM * ROW_LDS];
    alignas(16) int8_t b[BN_ROWS * ROW_LDS];
    alignas(16) float xs[GPC][BM];
    alignas(16) float ws[GPC][BN_ROWS];
};

// A group's operand fragments: lane (lr, h) holds bytes [16h, 16h + 16) of x
// row lr and of weight rows lr of the two tiles.
struct Frags {
    v4i a, b0, b1;
};

__device__ __forceinline__ void read_frags(const int8_t* la, const int8_t* lb0, const int8_t* lb1, int gi, Frags& f) {
    f.a = *(const v4i*)(la + 32 * gi);
    f.b0 = *(const v4i*)(lb0 + 32 * gi);
    f.b1 = *(const v4i*)(lb1 + 32 * gi);
}

// The i32 dots of a group for the wave's two weight tiles.
__device__ __forceinline__ void mfma_group(const Frags& f, v16i& d0, v16i& d1) {
    d0 = __builtin_amdgcn_mfma_i32_32x32x32_i8(f.a, f.b0, d0, 0, 0, 0);
    d1 = __builtin_amdgcn_mfma_i32_32x32x32_i8(f.a, f.b1, d1, 0, 0, 0);
}

// A group's scales for the lane: x scales of its 16 output rows (four
// runs of four), weight scales of its two columns.
struct Scales {
    float4 x[4];
    float w0, w1;
};

__device__ __forceinline__ void read_scales(const float* xs, const float* ws, int xrow, int c0, int c1, Scales& s) {
#pragma unroll
    for (int q = 0; q < 4; ++q) s.x[q] = *(const float4*)(xs + xrow + 8 * q);
    s.w0 = ws[c0];
    s.w1 = ws[c1];
}

// Q8_0 / Q4_K products of k not a multiple of 128.
template <int P, bool GELU>
__global__ __launch_bounds__(GEMM_THREADS, 2) void gemm_kernel(const int8_t* __restrict__ xq,
                                                               const float* __restrict__ xs, int m, int mpad,
                                                               const int8_t* __restrict__ codes,
                                                               const uint16_t* __restrict__ scales,
                                                               const float* __restrict__ bias, int n, int k,
                                                               int nb, int mb, GemvArgs a) {
    __shared__ __align__(16) Stage st;
    if (a.skip && *a.skip) return;
    // The last chunk holds k % KC bytes, zero past them, and chains only its
    // real groups.
    const int groups = k / 32, chunks = (k + KC - 1) / KC;
    // Tiles in XCD order: block b runs on XCD b % 8; the blocks of one XCD
    // share weight tiles, which then stay in that XCD's L2.
    const int blk = blockIdx.x;
    int bn, bm;
    if (nb % 8 == 0) {
        const int q = blk / 8;
        bn = blk % 8 + 8 * (q / mb);
        bm = q % mb;
    } else {
        bn = blk % nb;
        bm = blk / nb;
    }
    const int t = threadIdx.x;
    const int lane = t % WAVE, w = t / WAVE;
    const int lr = lane % 32, h = lane / 32;
    const int mbase = bm * BM;
    // LDS weight row i holds weight row brow(i): 128 rows, or for the
    // SwiGLU pair 64 gate rows then their 64 up rows.
    // Rows past n (the last tile when n % 128 != 0) load row n - 1 and
    // store nothing.
    auto brow = [&](int i) {
        const int r = P == 1 ? bn * 128 + i : (i < 64 ? bn * 64 + i : n / 2 + bn * 64 + (i - 64));
        return r < n ? r : n - 1;
    };

    // Global loads of a chunk, 16 bytes a piece, 16 threads a row (256
    // contiguous bytes): 4 x pieces and 8 weight pieces per thread; threads
    // [0, 16*GPC) one float4 of x scales, threads [128, 256) one weight row's
    // GPC scales.
    // Byte offsets of the thread's pieces in row 0 of the chunk; rows are
    // k bytes apart (x: at most m*k < 2^31 bytes, weights: n*k).
    uint32_t ag[4], bg[8];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int p = t + GEMM_THREADS * i, row = p / 16;
        const int mrow = mbase + row < m ? mbase + row : m - 1;
        ag[i] = (uint32_t)mrow * (uint32_t)k + 16 * (p % 16);
    }
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        const int p = t + GEMM_THREADS * i;
        bg[i] = (uint32_t)brow(p / 16) * (uint32_t)k + 16 * (p % 16);
    }
    const bool xs_thread = t < 16 * GPC;
    const bool ws_thread = t >= 128;
    const int ws_row = t - 128;
    const size_t ws_base = ws_thread ? (size_t)brow(ws_row) * groups : 0;

    v4i ra[4], rb[8];
    float4 rx = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    uint32_t rw[4] = {0, 0, 0, 0};  // 8 f16 scales
    auto fetch = [&](int c) {
        const size_t off = (size_t)c * KC;
        // Every piece of the thread sits at byte 16 (t % 16) of its row's chunk.
        const bool in_k = 16 * (t % 16) < k - c * KC;
#pragma unroll
        for (int i = 0; i < 4; ++i) ra[i] = in_k ? *(const v4i*)(xq + ag[i] + off) : v4i{0, 0, 0, 0};
#pragma unroll
        for (int i = 0; i < 8; ++i) rb[i] = in_k ? *(const v4i*)(codes + bg[i] + off) : v4i{0, 0, 0, 0};
        if (xs_thread) {
            if (c * GPC + t / 16 < groups)
                rx = *(const float4*)(xs + (size_t)(c * GPC + t / 16) * mpad + mbase + 4 * (t % 16));
            else
                rx = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        }
        if (ws_thread) {
            // A row's scales start anywhere: one load a scale, none past the row.
#pragma unroll
            for (int j = 0; j < GPC; ++j) {
                if (j % 2 == 0) rw[j / 2] = 0;
                if (c * GPC + j < groups) rw[j / 2] |= (uint32_t)scales[ws_base + c * GPC + j] << (16 * (j % 2));
            }
        }
    };
    auto stash = [&]() {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int p = t + GEMM_THREADS * i;
            *(v4i*)(st.a + (p / 16) * ROW_LDS + 16 * (p % 16)) = ra[i];
        }
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const int p = t + GEMM_THREADS * i;
            *(v4i*)(st.b + (p / 16) * ROW_LDS + 16 * (p % 16)) = rb[i];
        }
        if (xs_thread) *(float4*)(&st.xs[t / 16][4 * (t % 16)]) = rx;
        if (ws_thread) {
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                st.ws[2 * j][ws_row] = f16_to_f32((uint16_t)(rw[j] & 0xffff));
                st.ws[2 * j + 1][ws_row] = f16_to_f32((uint16_t)(rw[j] >> 16));
            }
        }
    };

    // The wave's tiles: x rows [32 (w % 2), +32) of the block; weight LDS
    // rows sub0 and sub1 (+32 each).
    const int wn = w / 2;
    const int sub0 = P == 1 ? wn * 64 : wn * 32;
    const int sub1 = P == 1 ? wn * 64 + 32 : 64 + wn * 32;
    const int8_t* la = st.a + ((w % 2) * 32 + lr) * ROW_LDS + 16 * h;
    const int8_t* lb0 = st.b + (sub0 + lr) * ROW_LDS + 16 * h;
    const int8_t* lb1 = st.b + (sub1 + lr) * ROW_LDS + 16 * h;
    const int xrow = (w % 2) * 32 + 4 * h;

    float t0[16], t1[16];
#pragma unroll
    for (int r = 0; r < 16; ++r) t0[r] = t1[r] = 0.0f;

    fetch(0);
    for (int c = 0; c < chunks; ++c) {
        __syncthreads();  // the previous chunk's reads are done
        stash();
        __syncthreads();
        if (c + 1 < chunks) fetch(c + 1);  // lands while this chunk computes
        // Software pipeline over the chunk's groups: at step gi the matrix
        // cores run group gi + 1 from fragments read one step earlier, LDS
        // reads for group gi + 2 are in flight, and the vector ALUs run
        // group gi's f32 chain. Scheduling barriers keep the compiler from
        // folding the stages back together.
        Frags f, fn;
        v16i d0 = {}, d1 = {};
        read_frags(la, lb0, lb1, 0, f);
        mfma_group(f, d0, d1);
        read_frags(la, lb0, lb1, 1, f);
#pragma unroll
        for (int gi = 0; gi < GPC; ++gi) {
            v16i n0 = {}, n1 = {};
            if (gi + 1 < GPC) mfma_group(f, n0, n1);
            if (gi + 2 < GPC) read_frags(la, lb0, lb1, gi + 2, fn);
            Scales sc;
            read_scales(st.xs[gi], st.ws[gi], xrow, sub0 + lr, sub1 + lr, sc);
            __builtin_amdgcn_sched_barrier(0);
            // Output (row 8*(r/4) + 4h + r%4, column lr) of a tile is register r.
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                if (c * GPC + gi >= groups) break;  // past k: no chain step
                const float xv[4] = {sc.x[q].x, sc.x[q].y, sc.x[q].z, sc.x[q].w};
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const int r = 4 * q + j;
                    t0[r] = __builtin_fmaf((float)d0[r], sc.w0 * xv[j], t0[r]);
                    t1[r] = __builtin_fmaf((float)d1[r], sc.w1 * xv[j], t1[r]);
                }
            }
            __builtin_amdgcn_sched_barrier(0);
            d0 = n0;
            d1 = n1;
            f = fn;
        }
    }

    // Epilogue, as the small-batch kernel's: bias, relu, then the residual
    // add or the SwiGLU pair (src/models/parts/causal_lm.rs:464-473).
    const int r0 = P == 1 ? bn * 128 + sub0 : bn * 64 + wn * 32;
    const int r1 = P == 1 ? bn * 128 + sub1 : n / 2 + r0;
    const int m0 = mbase + (w % 2) * 32;
    const int ldy = n / P;
#pragma unroll
    for (int r = 0; r < 16; ++r) {
        const int row = m0 + 8 * (r / 4) + 4 * h + r % 4;
        if (row >= m) continue;
        float v[2] = {t0[r], t1[r]};
        finish_outputs<GELU>(v, bias, {min(r0 + lr, n - 1), min(r1 + lr, n - 1)}, a.relu);  // columns past n are not stored
        if (P == 2) {
            a.y[(size_t)row * ldy + r0 + lr] = silu_trit(v[0]) * v[1];
            continue;
        }
        const size_t i0 = (size_t)row * ldy + r0 + lr, i1 = (size_t)row * ldy + r1 + lr;
        if (r0 + lr < n) a.y[i0] = a.epilogue == EPI_RESIDUAL ? a.residual[i0] + v[0] : v[0];
        if (r1 + lr < n) a.y[i1] = a.epilogue == EPI_RESIDUAL ? a.residual[i1] + v[1] : v[1];
    }
}

// The same product with the K stages loaded straight into LDS
// (global_load_lds_dwordx4: no staging registers) and double-buffered, so
// one barrier a stage suffices and several blocks share a CU: the vector
// ALUs, which bound this bit-exact product, stay busy while waves wait on
// LDS, the matrix cores or a barrier. A stage holds 128 bytes of K (four
// Q8_0 groups or one int8 group) of the block's 64 x rows and 64 TW weight
// rows, and the stage's scales as they lie in memory (x scales f32
// group-major, weight scales f16 or f32 per row). A row's eight 16-byte
// pieces sit in LDS in the order piece ^ ((row >> 1) & 7), so the 32 rows
// a wave's MFMA operand reads start in different banks. Waves 2 x 2: a wave
// owns 32 x rows by TW 32-row weight tiles (TW = 2: 128-row blocks, 3 a CU,
// 52 KB of LDS each; TW = 1: 64-row blocks, 4 a CU, 35 KB -- for products
// too narrow to give every CU the same number of wide blocks). The SwiGLU
// pair takes TW = 2 (a lane holds the gate and the up output it joins).
// k must be a multiple of 128.
constexpr int KD = 128;
typedef __attribute__((address_space(3))) void LdsVoid;

template <int TW>
struct alignas(16) DStage {
    alignas(16) int8_t a[BM * KD];
    alignas(16) int8_t b[64 * TW * KD];
    alignas(16) float xs[4 * BM];            // [group of the stage][x row]
    alignas(16) uint32_t ws[2 * 64 * TW];    // f16: row r's four at [2r, 2r + 2); f32: row r's one at [r]
};

__device__ __forceinline__ int piece_swizzle(int row) { return (row >> 1) & 7; }

// Loads of 16 (4) bytes a lane from g into LDS at l + 16 (4) x lane (l the
// same for the wave). Written out rather than as the compiler's builtin,
// whose wait counting, unable to tell the stages apart, can wait for every
// load in flight before a read of the other stage; the kernel waits for
// these loads itself (vmcnt).
__device__ __forceinline__ uint32_t lds_address(const void* l) { return (uint32_t)(uintptr_t)(const LdsVoid*)l; }

__device__ __forceinline__ void load16_to_lds(const void* g, void* l) {
    asm volatile("global_load_lds_dwordx4 %0, off" ::"v"(g), "{m0}"(lds_address(l)) : "memory");
}

__device__ __forceinline__ void load4_to_lds(const void* g, void* l) {
    asm volatile("global_load_lds_dword %0, off" ::"v"(g), "{m0}"(lds_address(l)) : "memory");
}

template <int G, bool HALF, int P, int TW, bool GELU>
__global__ __launch_bounds__(GEMM_THREADS, TW == 2 ? 3 : 4) void gemm_dma_kernel(
    const int8_t* __restrict__ xq, const float* __restrict__ xs, int m, int mpad, const int8_t* __restrict__ codes,
    const void* __restrict__ scales, const float* __restrict__ bias, int n, int k, int nb, int mb, GemvArgs a) {
    constexpr int GPC = KD / G;  // groups per stage
    constexpr int CH = G / 32;   // MFMA steps per group
    constexpr int BN = 64 * TW;  // weight rows per block
    static_assert(GPC * CH == 4, "a stage is four 32-byte MFMA steps");
    static_assert(P == 1 || TW == 2, "the SwiGLU pair: gate and up tiles in one wave");
    __shared__ DStage<TW> st0, st1;
    if (a.skip && *a.skip) return;
    const int groups = k / G, chunks = k / KD;
    const int blk = blockIdx.x;
    int bn, bm;
    if (nb % 8 == 0) {
        const int q = blk / 8;
        bn = blk % 8 + 8 * (q / mb);
        bm = q % mb;
    } else {
        bn = blk % nb;
        bm = blk / nb;
    }
    const int t = threadIdx.x;
    const int lane = t % WAVE, w = __builtin_amdgcn_readfirstlane(t / WAVE);
    const int lr = lane % 32, h = lane / 32;
    const int mbase = bm * BM;
    // LDS weight row i holds weight row brow(i); for the SwiGLU pair, 64
    // gate rows then their 64 up rows. Rows past n load row n - 1.
    auto brow = [&](int i) {
        const int r = P == 1 ? bn * BN + i : (i < 64 ? bn * 64 + i : n / 2 + bn * 64 + (i - 64));
        return r < n ? r : n - 1;
    };

    // The wave's loads of a stage: 1 KB an instruction (eight rows of 128
    // bytes), x rows [16w, +16) and weight rows [16 TW w, +16 TW); then SPW
    // scale loads: item 0 the x scales (1 KB: four groups of 64 rows, or one
    // group and copies), items 1.. the weight scales (f16: 32 rows an item,
    // two dwords a row; f32: 64 rows an item, one dword a row), items
    // w, w + 4, ... for wave w (a wave past the last item repeats it: the
    // same bytes to the same place).
    uint32_t ag[2], bg[2 * TW];
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        const int rl = 8 * (2 * w + i) + lane / 8;
        const int mrow = mbase + rl < m ? mbase + rl : m - 1;
        ag[i] = (uint32_t)mrow * (uint32_t)k + 16 * ((lane % 8) ^ piece_swizzle(rl));
    }
#pragma unroll
    for (int i = 0; i < 2 * TW; ++i) {
        const int rl = 8 * (2 * TW * w + i) + lane / 8;
        bg[i] = (uint32_t)brow(rl) * (uint32_t)k + 16 * ((lane % 8) ^ piece_swizzle(rl));
    }
    constexpr int NWS = HALF ? 2 * TW : TW;  // weight-scale items
    constexpr int SPW = (1 + NWS + 3) / 4;   // scale loads a wave
    int item[SPW];
    size_t soff[SPW];
#pragma unroll
    for (int j = 0; j < SPW; ++j) {
        const int it = w + 4 * j < 1 + NWS ? w + 4 * j : NWS;
        item[j] = it;
        if (it == 0)
            soff[j] = (size_t)(GPC == 4 ? lane / 16 : 0) * mpad + mbase + 4 * (lane % 16);
        else if (HALF)
            soff[j] = (size_t)brow(32 * (it - 1) + lane / 2) * (groups / 2) + lane % 2;
        else
            soff[j] = (size_t)brow(64 * (it - 1) + lane) * groups;
    }
    auto issue = [&](int c, DStage<TW>& s) {
        const size_t off = (size_t)c * KD;
#pragma unroll
        for (int i = 0; i < 2; ++i) load16_to_lds(xq + ag[i] + off, s.a + 1024 * (2 * w + i));
#pragma unroll
        for (int i = 0; i < 2 * TW; ++i) load16_to_lds(codes + bg[i] + off, s.b + 1024 * (2 * TW * w + i));
#pragma unroll
        for (int j = 0; j < SPW; ++j) {
            if (item[j] == 0)
                load16_to_lds(xs + soff[j] + (size_t)c * GPC * mpad, s.xs);
            else if (HALF)
                load4_to_lds((const uint32_t*)scales + soff[j] + 2 * c, s.ws + 64 * (item[j] - 1));
            else
                load4_to_lds((const float*)scales + soff[j] + c, s.ws + 64 * (item[j] - 1));
        }
    };

    // The wave's tiles: x rows [32 (w % 2), +32); weight LDS rows sub0 (and
    // sub1 for TW = 2), 32 each. Lane (lr, h) reads piece 2 s + h of its
    // rows for step s; its rows all share (lr >> 1) & 7.
    const int wn = w / 2;
    const int sub0 = TW == 1 ? wn * 32 : P == 1 ? wn * 64 : wn * 32;
    const int sub1 = TW == 1 ? sub0 : P == 1 ? wn * 64 + 32 : 64 + wn * 32;
    uint32_t pa[4], pb[4];
#pragma unroll
    for (int s4 = 0; s4 < 4; ++s4) {
        const int po = 16 * ((2 * s4 + h) ^ piece_swizzle(lr));
        pa[s4] = ((w % 2) * 32 + lr) * KD + po;
        pb[s4] = (sub0 + lr) * KD + po;
    }
    constexpr int B1 = (P == 1 ? 32 : 64) * KD;  // sub1 - sub0 rows, in bytes (TW = 2)

    float t0[16], t1[16];
#pragma unroll
    for (int r = 0; r < 16; ++r) t0[r] = t1[r] = 0.0f;

    // The scale products come from the matrix cores: the outer product of 32 x
    // scales and 32 weight scales in the dots' register layout, each
    // fma(xs, ws, 0), which is the vector multiply's one rounding.
    // v_mfma_f32_32x32x1_2b makes two of them, of a tile's two groups (TW = 1)
    // or of the two tiles (TW = 2), half h of the lanes giving the second's
    // scales. LDS bounded the kernel, most of it the sixteen x scales a lane
    // read for the multiply; the outer product reads one (time in indexed LDS
    // access, SQ_LDS_IDX_ACTIVE, 5.02 M to 2.25 M a dispatch of 1564 x 2048 x
    // 2048, of 12 M busy CU cycles). The conversions of two tiles go before their multiply-adds:
    // a dependent vector instruction costs 10.5 cycles, and without the
    // scheduling barriers the compiler pairs each multiply-add with the
    // conversion just before it (in that order the outer product was slower
    // than the multiply: 55 us a 1564-row product against 46). The three
    // products of a 1564-row prompt (n 2048, 6144, 2048; k 2048): 139 -> 126 us.
    const v16i magic = dot_base();
    const int xr = (w % 2) * 32 + lr, wr = TW == 1 ? sub0 + lr : (h ? sub1 : sub0) + lr;
    auto weight_scale = [&](const DStage<TW>& s, int g) {
        if (HALF) return f16_to_f32(((const uint16_t*)s.ws)[4 * wr + g]);
        return __builtin_bit_cast(float, s.ws[wr]);
    };
    auto compute = [&](const DStage<TW>& s) {
        const int8_t* sa = s.a;
        const int8_t* sb = s.b;
        auto dots = [&](int g, int tile) {
            v16i d = magic;
#pragma unroll
            for (int c4 = 0; c4 < CH; ++c4) {
                const int s4 = g * CH + c4;
                d = __builtin_amdgcn_mfma_i32_32x32x32_i8(*(const v4i*)(sa + pa[s4]),
                                                          *(const v4i*)(sb + pb[s4] + tile * B1), d, 0, 0, 0);
            }
            return d;
        };
        // Two dots' chain steps: all the conversions, then the multiply-adds.
        auto chain2 = [&](float (&ta)[16], float (&tb)[16], const v16i& d0, const v16i& d1, const v32f& sc) {
            float f0[16], f1[16];
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int r = 0; r < 16; ++r) f0[r] = dot_of(d0[r]);
#pragma unroll
            for (int r = 0; r < 16; ++r) f1[r] = dot_of(d1[r]);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int r = 0; r < 16; ++r) ta[r] = __builtin_fmaf(f0[r], sc[r], ta[r]);
#pragma unroll
            for (int r = 0; r < 16; ++r) tb[r] = __builtin_fmaf(f1[r], sc[16 + r], tb[r]);
            __builtin_amdgcn_sched_barrier(0);
        };
        if constexpr (TW == 2) {
#pragma unroll
            for (int g = 0; g < GPC; ++g) {
                const v32f sc = __builtin_amdgcn_mfma_f32_32x32x1f32(s.xs[g * BM + xr], weight_scale(s, g), v32f{}, 0, 0, 0);
                const v16i d0 = dots(g, 0), d1 = dots(g, 1);
                chain2(t0, t1, d0, d1, sc);
            }
        } else if constexpr (GPC > 1) {
#pragma unroll
            for (int g = 0; g < GPC; g += 2) {
                const v32f sc = __builtin_amdgcn_mfma_f32_32x32x1f32(s.xs[(g + h) * BM + xr], weight_scale(s, g + h), v32f{}, 0, 0, 0);
                const v16i d0 = dots(g, 0), d1 = dots(g + 1, 0);
                chain2(t0, t0, d0, d1, sc);
            }
        } else {
            // One group a stage: the vector ALUs make the scale products (of the
            // outer product half would go unused: 1564 rows of 2651x512 16.2 us
            // against 16.4, of 6144x2048 57.8 against 58.8, fewer rows the same).
            const float wv = weight_scale(s, 0);
            const v16i d = dots(0, 0);
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const float4 x4 = *(const float4*)(s.xs + (w % 2) * 32 + 4 * h + 8 * q);
                const float xv[4] = {x4.x, x4.y, x4.z, x4.w};
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const int r = 4 * q + j;
                    t0[r] = __builtin_fmaf(dot_of(d[r]), wv * xv[j], t0[r]);
                }
            }
        }
    };

    // Two stages: stage c + 1 loads while stage c computes. (A third stage
    // in flight, with a block fewer a CU for its LDS, measured slower.)
    auto step = [&](int c, DStage<TW>& cur, DStage<TW>& next) {
        // This wave's loads of stage c (the only ones in flight) landed; the
        // barrier: every wave's, and every wave is done with stage c - 1,
        // whose buffer stage c + 1 takes. A bare barrier: __syncthreads
        // would add nothing the wait does not already give.
        __builtin_amdgcn_s_waitcnt(0x0f70);  // vmcnt(0)
        asm volatile("s_barrier" ::: "memory");
        if (c + 1 < chunks) issue(c + 1, next);
        compute(cur);
    };
    issue(0, st0);
    for (int c = 0; c < chunks; c += 2) {
        step(c, st0, st1);
        if (c + 1 >= chunks) break;
        step(c + 1, st1, st0);
    }

    // Epilogue, as gemm_kernel's (src/models/parts/causal_lm.rs:464-473).
    const int r0 = P == 1 ? bn * BN + sub0 : bn * 64 + wn * 32;
    const int r1 = P == 1 ? bn * BN + sub1 : n / 2 + r0;
    const int m0 = mbase + (w % 2) * 32;
    const int ldy = n / P;
#pragma unroll
    for (int r = 0; r < 16; ++r) {
        const int row = m0 + 8 * (r / 4) + 4 * h + r % 4;
        if (row >= m) continue;
        float v[TW] = {t0[r]};
        int col[TW] = {min(r0 + lr, n - 1)};
        if constexpr (TW == 2) {
            v[1] = t1[r];
            col[1] = min(r1 + lr, n - 1);
        }
        finish_outputs<GELU>(v, bias, col, a.relu);
        if constexpr (P == 2) {
            a.y[(size_t)row * ldy + r0 + lr] = silu_trit(v[0]) * v[1];
            continue;
        }
        const size_t i0 = (size_t)row * ldy + r0 + lr;
        if (r0 + lr < n) a.y[i0] = a.epilogue == EPI_RESIDUAL ? a.residual[i0] + v[0] : v[0];
        if constexpr (TW == 2) {
            const size_t i1 = (size_t)row * ldy + r1 + lr;
            if (r1 + lr < n) a.y[i1] = a.epilogue == EPI_RESIDUAL ? a.residual[i1] + v[1] : v[1];
        }
    }
}

// Large Q8_0 / Q4_K products of k not a multiple of 128 (an ASR stem's 4320-input
// convolutions): 128 x rows by 128 weight rows a block, stages as above, two
// blocks a CU by their LDS (73 KB). A wave owns 64 x 64 outputs as 2 x 2 MFMA
// tiles, so a byte loaded and a byte read from LDS feed twice the outputs of
// the 64 x 64 blocks, in half the waves. Scale products and conversions as
// above. The last stage's pieces past k load the row's first piece of the
// stage, its groups past k are not chained, and a row's four f16 scales, which
// start at any 2-byte offset, are loaded as the three dwords that hold them.
struct alignas(16) WStage {
    alignas(16) int8_t a[128 * KD];
    alignas(16) int8_t b[128 * KD];
    alignas(16) float xs[4 * 128];  // [group of the stage][x row]
    alignas(16) uint32_t ws[3 * 128];
};

template <bool GELU>
__global__ __launch_bounds__(GEMM_THREADS, 2) void gemm_wide_kernel(
    const int8_t* __restrict__ xq, const float* __restrict__ xs, int m, int mpad, const int8_t* __restrict__ codes,
    const void* __restrict__ scales, const float* __restrict__ bias, int n, int k, int nb, int mb, GemvArgs a) {
    __shared__ WStage st0, st1;
    if (a.skip && *a.skip) return;
    const int groups = k / 32, chunks = (k + KD - 1) / KD;
    const int blk = blockIdx.x;
    int bn, bm;
    if (nb % 8 == 0) {
        const int q = blk / 8;
        bn = blk % 8 + 8 * (q / mb);
        bm = q % mb;
    } else {
        bn = blk % nb;
        bm = blk / nb;
    }
    const int t = threadIdx.x;
    const int lane = t % WAVE, w = __builtin_amdgcn_readfirstlane(t / WAVE);
    const int lr = lane % 32, h = lane / 32;
    const int mbase = bm * 128;
    // LDS weight row i holds weight row brow(i); rows past n load row n - 1.
    auto brow = [&](int i) { return min(bn * 128 + i, n - 1); };

    // The wave's loads of a stage: x rows and weight rows [32 w, +32), 1 KB
    // (eight rows of 128 bytes) an instruction; then scale items w and w + 4
    // (x scales, 16 bytes a lane; weight scales, a dword a lane).
    uint32_t ag[4], bg[4], piece[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int rl = 8 * (4 * w + i) + lane / 8;
        piece[i] = 16 * ((lane % 8) ^ piece_swizzle(rl));
        ag[i] = (uint32_t)(mbase + rl < m ? mbase + rl : m - 1) * (uint32_t)k;
        bg[i] = (uint32_t)brow(rl) * (uint32_t)k;
    }
    // Items 0 and 1 are the x scales of two groups each, 2 .. 7 the weight
    // rows' scale dwords.
    int item[2];
    size_t soff[2];
#pragma unroll
    for (int j = 0; j < 2; ++j) {
        item[j] = w + 4 * j;
        const int d = 64 * (item[j] - 2) + lane;
        // x rows past mpad (none of them stored) take its last four.
        soff[j] = item[j] < 2 ? (size_t)min(mbase + 4 * (lane % 32), mpad - 4)
                              : ((size_t)brow(d / 3) * groups) / 2 + d % 3;
    }
    const size_t last_dword = ((size_t)n * groups - 1) / 2;
    auto issue = [&](int c, WStage& s) {
        const size_t off = (size_t)c * KD;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const uint32_t p = (int)(off + piece[i]) < k ? piece[i] : 0;
            load16_to_lds(xq + ag[i] + off + p, s.a + 1024 * (4 * w + i));
            load16_to_lds(codes + bg[i] + off + p, s.b + 1024 * (4 * w + i));
        }
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            if (item[j] < 2) {
                const int g = min(4 * c + 2 * item[j] + lane / 32, groups - 1);
                load16_to_lds(xs + soff[j] + (size_t)g * mpad, s.xs + 256 * item[j]);
            } else {
                load4_to_lds((const uint32_t*)scales + min(soff[j] + 2 * c, last_dword), s.ws + 64 * (item[j] - 2));
            }
        }
    };

    // The wave's tiles: x rows [64 (w % 2), +64) of the block, weight LDS rows
    // sub0 and sub1, 32 each. Lane (lr, h) reads piece 2 s + h of its rows for
    // step s; its rows all share (lr >> 1) & 7.
    const int wn = w / 2;
    const int sub0 = wn * 64, sub1 = sub0 + 32;
    const int xr = (w % 2) * 64 + lr, wr = (h ? sub1 : sub0) + lr;
    uint32_t pa[4], pb[4];
#pragma unroll
    for (int s4 = 0; s4 < 4; ++s4) {
        const int po = 16 * ((2 * s4 + h) ^ piece_swizzle(lr));
        pa[s4] = xr * KD + po;
        pb[s4] = (sub0 + lr) * KD + po;
    }
    constexpr int T1 = 32 * KD;  // a tile
    // Half h of the lanes holds the scales of tile h: their first's offset in the three dwords.
    const int wodd = (int)(((size_t)brow(wr) * groups) & 1);
    const v16i magic = dot_base();
    float acc[2][2][16];
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.0f;

    auto compute = [&](const WStage& s, int c) {
#pragma unroll
        for (int g = 0; g < 4; ++g) {
            if (4 * c + g >= groups) break;
            const float wv = f16_to_f32(((const uint16_t*)s.ws)[6 * wr + wodd + g]);
            const v4i fa[2] = {*(const v4i*)(s.a + pa[g]), *(const v4i*)(s.a + pa[g] + T1)};
            const v4i fb[2] = {*(const v4i*)(s.b + pb[g]), *(const v4i*)(s.b + pb[g] + T1)};
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                const v32f sc = __builtin_amdgcn_mfma_f32_32x32x1f32(s.xs[g * 128 + xr + 32 * i], wv, v32f{}, 0, 0, 0);
                v16i d[2];
#pragma unroll
                for (int j = 0; j < 2; ++j) d[j] = __builtin_amdgcn_mfma_i32_32x32x32_i8(fa[i], fb[j], magic, 0, 0, 0);
                // Output (row 8*(r/4) + 4h + r%4, column lr) of a tile is register r.
                // Conversions first, as in the kernel above.
                float f[2][16];
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int j = 0; j < 2; ++j)
#pragma unroll
                    for (int r = 0; r < 16; ++r) f[j][r] = dot_of(d[j][r]);
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int j = 0; j < 2; ++j)
#pragma unroll
                    for (int r = 0; r < 16; ++r)
                        acc[i][j][r] = __builtin_fmaf(f[j][r], sc[16 * j + r], acc[i][j][r]);
            }
        }
    };

    // Two stages: stage c + 1 loads while stage c computes.
    auto step = [&](int c, WStage& cur, WStage& next) {
        // This wave's loads of stage c (the only ones in flight) landed; the
        // barrier: every wave's, and every wave is done with stage c - 1,
        // whose buffer stage c + 1 takes.
        __builtin_amdgcn_s_waitcnt(0x0f70);  // vmcnt(0)
        asm volatile("s_barrier" ::: "memory");
        if (c + 1 < chunks) issue(c + 1, next);
        compute(cur, c);
    };
    issue(0, st0);
    for (int c = 0; c < chunks; c += 2) {
        step(c, st0, st1);
        if (c + 1 >= chunks) break;
        step(c + 1, st1, st0);
    }

    // Epilogue, as gemm_kernel's (src/models/parts/causal_lm.rs:464-473).
    const int r0 = bn * 128 + sub0, r1 = r0 + 32;
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            const int row = mbase + (w % 2) * 64 + 32 * i + 8 * (r / 4) + 4 * h + r % 4;
            if (row >= m) continue;
            float v[2] = {acc[i][0][r], acc[i][1][r]};
            finish_outputs<GELU>(v, bias, {min(r0 + lr, n - 1), min(r1 + lr, n - 1)}, a.relu);
            const size_t i0 = (size_t)row * n + r0 + lr, i1 = (size_t)row * n + r1 + lr;
            if (r0 + lr < n) a.y[i0] = a.epilogue == EPI_RESIDUAL ? a.residual[i0] + v[0] : v[0];
            if (r1 + lr < n) a.y[i1] = a.epilogue == EPI_RESIDUAL ? a.residual[i1] + v[1] : v[1];
        }
}

// Ternary products of many rows: 2-bit codes, f32 scales a 128-group, the
// same contract (dot of the codes minus one and the activation codes). A wave
// owns 32 x rows by TN 32-row weight tiles, four waves a block (2 x 2); no LDS
// and no barriers, every operand straight from global memory, four groups in
// flight: what bounds it is the address lines of the loads, so the codes of x
// are quantized into operand order (ternary_code) and the weight scales load
// four groups at once (from row-major codes, each load touching 32 rows, 375
// rows through 4096 x 1024 and 1024 x 4096 took 48 us; 37 us so). The order of
// K inside a group is free (an integer dot): MFMA step s
// of a group takes the codes 64 h + 16 s .. + 15 for the half h of the lanes,
// so a lane's 16 bytes of 2-bit codes are its four steps' operands, each dword
// unpacked by shifts, a mask and a byte permute that looks up code - 1. The
// scale products ws * xs come from the matrix cores as well, the outer product
// of the two scale vectors in the dots' register layout (one product rounded
// once, as the vector multiply rounds it), which leaves a conversion and a
// multiply-add an output to the vector ALUs.
constexpr int TERN_DEPTH = 4;

template <int TN, bool GELU>
__global__ __launch_bounds__(GEMM_THREADS, 2) void gemm_ternary_kernel(const int8_t* __restrict__ xq,
                                                                       const float* __restrict__ xs, int m, int mpad,
                                                                       const uint8_t* __restrict__ codes,
                                                                       const float* __restrict__ scales,
                                                                       const float* __restrict__ bias, int n, int k,
                                                                       int nb, int mb, GemvArgs a) {
    if (a.skip && *a.skip) return;
    const int groups = k / 128;
    const int blk = blockIdx.x;
    int bn, bm;
    if (nb % 8 == 0) {
        const int q = blk / 8;
        bn = blk % 8 + 8 * (q / mb);
        bm = q % mb;
    } else {
        bn = blk % nb;
        bm = blk / nb;
    }
    const int lane = threadIdx.x % WAVE, w = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE);
    const int lr = lane % 32, h = lane / 32;
    const int m0 = bm * BM + 32 * (w % 2), n0 = (bn * 2 + w / 2) * 32 * TN;
    if (m0 >= m || n0 >= n) return;
    const int8_t* xp = xq + (size_t)(m0 / 32) * groups * 4096 + lane * 16;  // (rows past m: not stored)
    const float* xsp = xs + m0 + lr;  // mpad covers the tile's rows
    const uint8_t* wp[TN];
#pragma unroll
    for (int j = 0; j < TN; ++j) wp[j] = codes + (size_t)min(n0 + 32 * j + lr, n - 1) * (k / 4) + 16 * h;
    // The lane's weight scales: of row lr of tile h (TN = 2) or of the tile.
    const float* wsp = scales + (size_t)min(n0 + 32 * (TN == 2 ? h : 0) + lr, n - 1) * groups;
    v4i av[TERN_DEPTH][4];
    uint4 bv[TERN_DEPTH][TN];
    float xv[TERN_DEPTH], wv[TERN_DEPTH], wnext[TERN_DEPTH];
    auto fetch = [&](int g, int d) {
#pragma unroll
        for (int s = 0; s < 4; ++s) av[d][s] = *(const v4i*)(xp + (size_t)g * 4096 + 1024 * s);
        xv[d] = xsp[(size_t)g * mpad];
#pragma unroll
        for (int j = 0; j < TN; ++j) bv[d][j] = *(const uint4*)(wp[j] + (size_t)g * 32);
    };
    // The scales of groups g .. g + 3 (past the last: the last's again, not used).
    static_assert(TERN_DEPTH == 4, "four groups' scales a load");
    auto fetch_scales = [&](int g) {
        if (groups % 4 == 0) {
            const float4 f = *(const float4*)(wsp + min(g, groups - 4));
            wnext[0] = f.x;
            wnext[1] = f.y;
            wnext[2] = f.z;
            wnext[3] = f.w;
        } else {
#pragma unroll
            for (int d = 0; d < TERN_DEPTH; ++d) wnext[d] = wsp[min(g + d, groups - 1)];
        }
    };
    const v16i magic = dot_base();
    float t[TN][16];
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
        for (int r = 0; r < 16; ++r) t[j][r] = 0.0f;
#pragma unroll
    for (int d = 0; d < TERN_DEPTH; ++d)
        if (d < groups) fetch(d, d);
    fetch_scales(0);
    for (int g0 = 0; g0 < groups; g0 += TERN_DEPTH) {
#pragma unroll
        for (int d = 0; d < TERN_DEPTH; ++d) wv[d] = wnext[d];
        fetch_scales(g0 + TERN_DEPTH);
#pragma unroll
        for (int d = 0; d < TERN_DEPTH; ++d) {
            const int g = g0 + d;
            if (g >= groups) break;
            v16i dot[TN];
            v16f sc[TN];
            if constexpr (TN == 2) {
                const v32f both = __builtin_amdgcn_mfma_f32_32x32x1f32(xv[d], wv[d], v32f{}, 0, 0, 0);
                sc[0] = lower(both);
                sc[1] = upper(both);
            } else {
                sc[0] = __builtin_amdgcn_mfma_f32_32x32x2f32(h ? 0.0f : xv[d], h ? 0.0f : wv[d], v16f{}, 0, 0, 0);
            }
#pragma unroll
            for (int j = 0; j < TN; ++j) {
                const uint32_t words[4] = {bv[d][j].x, bv[d][j].y, bv[d][j].z, bv[d][j].w};
                dot[j] = magic;
#pragma unroll
                for (int s = 0; s < 4; ++s) {
                    v4i b;
#pragma unroll
                    for (int i = 0; i < 4; ++i)
                        b[i] = (int)__builtin_amdgcn_perm(0u, 0x020100FFu, (words[s] >> (2 * i)) & 0x03030303u);
                    dot[j] = __builtin_amdgcn_mfma_i32_32x32x32_i8(av[d][s], b, dot[j], 0, 0, 0);
                }
            }
            if (g + TERN_DEPTH < groups) fetch(g + TERN_DEPTH, d);
#pragma unroll
            for (int j = 0; j < TN; ++j)
#pragma unroll
                for (int r = 0; r < 16; ++r) t[j][r] = __builtin_fmaf(dot_of(dot[j][r]), sc[j][r], t[j][r]);
        }
    }
#pragma unroll
    for (int j = 0; j < TN; ++j) {
        const int col = n0 + 32 * j + lr;
        if (col >= n) continue;
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            const int row = m0 + 8 * (r / 4) + 4 * h + r % 4;
            if (row >= m) continue;
            float v[1] = {t[j][r]};
            finish_outputs<GELU>(v, bias, {col}, a.relu);
            const size_t at = (size_t)row * n + col;
            a.y[at] = a.epilogue == EPI_RESIDUAL ? a.residual[at] + v[0] : v[0];
        }
    }
}

// Whether 64-row weight blocks (four a CU) spread the product more evenly
// than 128-row ones (three a CU) -- TRIT_HIP_GEMM_TILE=64 or 128 forces one.
bool narrow(int n, int mb) {
    static const int forced = [] {
        const char* v = getenv("TRIT_HIP_GEMM_TILE");
        return v && *v ? (int)strtol(v, nullptr, 10) : 0;
    }();
    if (forced) return forced == 64;
    return true;
}

// Whether a plain product takes gemm_wide_kernel: k not a multiple of 128, and
// more 128 x 128 blocks than gemm_kernel's, two a CU, hold at once (256: past
// them that kernel starts a second wave of blocks), or rows long enough that half the
// loads a byte pay earlier. gemm_kernel against it, us (quantizer included): n
// 480, 384 blocks, k 32 15.8, 13.1, k 1056 61.7, 48.9, k 4320 244, 157; 192
// blocks, k 160 13.2, 14.7, k 1056 35.4, 35.3, k 2080 58.3, 57.1, k 4320 119,
// 105; one block row of at most 64 rows (half of each block unused), n 20480, 160
// blocks, k 1056 23.2, 26.8, k 2080 38.4, 42.9, k 3104 64.3, 58.3. For k a
// multiple of 128 the 64 x 64 blocks are faster (1564 x 6144 x 2048, 624 blocks:
// 68 us against 82).
bool wide(int nb, int m, int k) {
    const int64_t blocks = (int64_t)nb * ((m + 127) / 128);
    return k % KD != 0 && (blocks > 256 || (blocks >= 160 && k >= (m > 64 ? 2048 : 3072)));
}

template <int G, bool HALF, int P, bool GELU>
void launch_gemm(const Layer& L, const GemvArgs& a, const GemmScratch& sc, hipStream_t s) {
    const int nb = P == 1 ? (L.n + 127) / 128 : (L.n / 2) / 64;
    const int mb = sc.mpad / BM;
    if constexpr (G == 32 && P == 1) {
        if (wide(nb, a.m, L.k)) {
            const int mb2 = (a.m + 127) / 128;
            launch_timed(a, gemm_wide_kernel<GELU>, dim3(nb * mb2), dim3(GEMM_THREADS), 0, s, (const int8_t*)sc.xq,
                         (const float*)sc.xs, a.m, sc.mpad, L.codes.as<int8_t>(), (const void*)L.scales.ptr,
                         L.bias.as<float>(), L.n, L.k, nb, mb2, a);
            TRIT_HIP(hipGetLastError());
            return;
        }
    }
    if constexpr (P == 1) {
        if (L.k % KD == 0 && narrow(L.n, mb)) {
            const int nb1 = (L.n + 63) / 64;
            launch_timed(a, gemm_dma_kernel<G, HALF, P, 1, GELU>, dim3(nb1 * mb), dim3(GEMM_THREADS), 0, s,
                         (const int8_t*)sc.xq, (const float*)sc.xs, a.m, sc.mpad, L.codes.as<int8_t>(),
                         (const void*)L.scales.ptr, L.bias.as<float>(), L.n, L.k, nb1, mb, a);
            TRIT_HIP(hipGetLastError());
            return;
        }
    }
    if (L.k % KD == 0)
        launch_timed(a, gemm_dma_kernel<G, HALF, P, 2, GELU>, dim3(nb * mb), dim3(GEMM_THREADS), 0, s,
                     (const int8_t*)sc.xq, (const float*)sc.xs, a.m, sc.mpad, L.codes.as<int8_t>(),
                     (const void*)L.scales.ptr, L.bias.as<float>(), L.n, L.k, nb, mb, a);
    else if constexpr (G == 32)
        launch_timed(a, gemm_kernel<P, GELU>, dim3(nb * mb), dim3(GEMM_THREADS), 0, s,
                     (const int8_t*)sc.xq, (const float*)sc.xs, a.m, sc.mpad, L.codes.as<int8_t>(),
                     L.scales.as<uint16_t>(), L.bias.as<float>(), L.n, L.k, nb, mb, a);
    TRIT_HIP(hipGetLastError());
}

// Two weight tiles a wave from 192 blocks of them, else one: fewer leave CUs
// without a block. One tile against two, us (quantizer included), by the blocks
// of two: 1024x4096 128 28.0, 33.8, 192 39.4, 34.5, 256 41.6, 36.8; 4096x1024 64
// 9.8, 12.5, 192 14.1, 13.7, 1024 40.9, 34.9; 2048x2048 128 15.0, 18.7, 192 22.3,
// 20.6.
template <bool GELU>
void launch_ternary(const Layer& L, const GemvArgs& a, const GemmScratch& sc, hipStream_t s) {
    const int mb = sc.mpad / BM;
    auto go = [&](auto TN_) {
        constexpr int TN = decltype(TN_)::value;
        const int nb = (L.n + 64 * TN - 1) / (64 * TN);
        launch_timed(a, gemm_ternary_kernel<TN, GELU>, dim3(nb * mb), dim3(GEMM_THREADS), 0, s, (const int8_t*)sc.xq,
                     (const float*)sc.xs, a.m, sc.mpad, L.codes.as<uint8_t>(), L.scales.as<float>(),
                     L.bias.as<float>(), L.n, L.k, nb, mb, a);
    };
    if ((int64_t)((L.n + 127) / 128) * mb >= 192) go(std::integral_constant<int, 2>{});
    else go(std::integral_constant<int, 1>{});
    TRIT_HIP(hipGetLastError());
}

// The product of rows quantized into `sc`, with or without the GELU in its
// store.
template <bool GELU>
void launch_product(const Layer& L, const GemvArgs& a, const GemmScratch& sc, hipStream_t s) {
    if (L.kind == TERNARY) return launch_ternary<GELU>(L, a, sc, s);
    const bool int8 = L.kind == INT8;
    if constexpr (!GELU) {
        if (a.epilogue == EPI_SILU_PAIR)
            return int8 ? launch_gemm<128, false, 2, false>(L, a, sc, s) : launch_gemm<32, true, 2, false>(L, a, sc, s);
    }
    return int8 ? launch_gemm<128, false, 1, GELU>(L, a, sc, s) : launch_gemm<32, true, 1, GELU>(L, a, sc, s);
}

}  // namespace
}  // namespace trit
