// Exact FP8 products of several inputs on f32 matrix instructions with
// one term a step: the order of gemv_fp8_e4m3_ue8m0_rows_multi (E/compute.rs:
// 6384-6577) - per AVX lane l and 128-column group the chains g0 and g1 of
// eight FMAs (columns 16c + l and 16c + 8 + l), acc = fma(g0 + g1, scale,
// acc) over the groups, then the pairwise sum over l - bit for bit.
//
// v_mfma_f32_16x16x1_4b_f32 is four independent blocks of 16 x 16 outer
// products, D = A B + C with one product per output: an FMA rounded once, as
// v_fma_f32 (checked bit for bit over normal, tiny and infinite inputs).  So
// a block carries one chain of 16 rows x 16 inputs, and eight steps make
// eight FMAs of its chain.  The four blocks of a wave are the chains (l, g0),
// (l, g1), (l + 1, g0), (l + 1, g1) with l = 2 wave: g0 + g1, the scale and
// the accumulation over the groups stay in a lane, the four waves of a
// workgroup meet once, at the pairwise sum.
//
// Why: the vector kernel (k_fp8_gemv_multi) issues one FMA per 64 products,
// a decoded weight's register read again for every input: 512 products of a
// wave in the time a matrix instruction does 1024, and its LDS reads beside
// them.  13 inputs of a layer's five projections: 103.9 -> 85.6 us,
// of the 4096 x 8192 one 36.2 -> 22.2 us (6.8 us of matrix time; the rest is
// one wave a SIMD that also decodes, stages x and waits for the barriers).
#pragma once
#include "fp8_multi.h"

#define WH_FP8_XMM_GROUPS 4u  // 128-column groups a chunk of x in LDS
typedef float wh_f16 __attribute__((ext_vector_type(16)));

// Grid (blocks of 16 kT rows [+ the second tensor's], ceil(n_in / 16)), 256
// threads.  cols % 1024 == 0; row starts and rows per scale row are multiples
// of 16, rows of an input group of 16 kT (host checks).  A wave carries kT
// tiles of 16 rows, which halves the reads of x where that still leaves a
// workgroup for every CU.
template <bool kSpecial, bool kScaleU8, int kT>
__global__ void __launch_bounds__(256, 2) k_fp8_exact_mm(wh_fp8_args a, uint32_t n_in) {
    constexpr uint32_t kG = WH_FP8_XMM_GROUPS, kChunk = 128 * kG;
    constexpr uint32_t kLd = kChunk + 4;  // floats per input: 16 inputs' 16-byte reads fall on 16 bank groups
    constexpr int kUnits = 16 * kChunk / 16 / 256;
    __shared__ __align__(16) float xs[2][16 * kLd];
    extern __shared__ __align__(16) float scale_s[];  // [kT][cols / 128]
    const uint32_t t = threadIdx.x, wave = t >> 6, lane = t & 63, q = lane >> 4, col = lane & 15;
    const bool two = blockIdx.x >= a.blocks1;
    const uint8_t* w = two ? a.w2 : a.w;
    const void* sc = two ? a.scales2 : a.scales;
    const uint32_t scale_cols = two ? a.scale_cols2 : a.scale_cols;
    const uint32_t rg_shift = two ? a.row_group_shift2 : a.row_group_shift;
    const uint32_t r_lo = two ? a.row_start2 : a.row_start, r_hi = two ? a.row_end2 : a.row_end;
    float* yb = two ? a.y2 : a.y;
    const uint32_t row0 = r_lo + (two ? blockIdx.x - a.blocks1 : blockIdx.x) * (16 * kT);
    const uint32_t cols = a.cols, n_chunks = cols / kChunk;
    const uint32_t i0 = blockIdx.y * 16, n_here = min(16u, n_in - i0);
    const uint32_t grp = a.x_group_shift < 32 ? (row0 - a.row_start) >> a.x_group_shift : 0u;
    const float* xbase = a.x + (size_t)i0 * a.x_stride + (size_t)grp * a.x_group_stride;

    // A: block q = (l, half) of row `col`: the half's eight bytes of lane l
    const uint8_t* wp[kT];
#pragma unroll
    for (int i = 0; i < kT; ++i) {
        const uint32_t rt = row0 + 16 * i;
        wp[i] = w + (size_t)min(rt + col, r_hi - 1) * cols + 16 * (2 * wave + (q >> 1)) + 8 * (q & 1);
        // 16 rows of a tile share a scale row; its scales go to LDS first (a
        // scalar load in the loop is waited for with every LDS read after it)
        const uint32_t srow = (min(rt, r_hi - 1) >> rg_shift) * scale_cols;
        for (uint32_t g = t; g < cols / 128; g += 256)
            scale_s[i * (cols / 128) + g] = wh_fp8_scale<kSpecial, kScaleU8>(sc, srow + g);
    }
    uint2 wv[2][kT][kG];
    auto load_w = [&](int b, uint32_t chunk) {
        const uint32_t g0 = min(chunk, n_chunks - 1) * kG;
#pragma unroll
        for (int i = 0; i < kT; ++i)
#pragma unroll
            for (uint32_t g = 0; g < kG; ++g) wv[b][i][g] = *(const uint2*)(wp[i] + 128 * (g0 + g));
    };
    // x: unit u is 16 columns c of group g of input n, spread over the chains
    // (l, half), whose eight values are contiguous
    const uint32_t uc = t & 7, un = (t >> 3) & 15, ug = t >> 7;
    const float* xp = xbase + (size_t)min(un, n_here - 1) * a.x_stride + 128 * ug + 16 * uc;
    float4 xr[2][kUnits][4];
    auto load_x = [&](int b, uint32_t chunk) {
        const float* p = xp + (size_t)min(chunk, n_chunks - 1) * kChunk;
#pragma unroll
        for (int k = 0; k < kUnits; ++k)
#pragma unroll
            for (int j = 0; j < 4; ++j) xr[b][k][j] = *(const float4*)(p + 256 * k + 4 * j);
    };
    auto store_x = [&](int b) {
#pragma unroll
        for (int k = 0; k < kUnits; ++k) {
            float* d = xs[b] + un * kLd + 128 * (ug + 2 * k) + uc;
#pragma unroll
            for (int o = 0; o < 16; ++o) d[((o & 7) * 2 + (o >> 3)) * 8] = wh_f4_get(xr[b][k][o >> 2], o & 3);
        }
    };
    float acc[kT][2][4];
#pragma unroll
    for (int i = 0; i < kT; ++i)
#pragma unroll
        for (int l = 0; l < 2; ++l)
#pragma unroll
            for (int r = 0; r < 4; ++r) acc[i][l][r] = 0.0f;
    const float* xq = xs[0] + col * kLd + (4 * wave + q) * 8;
    auto chunk_mm = [&](int b, uint32_t k) {
#pragma unroll
        for (uint32_t g = 0; g < kG; ++g) {
            const float4* p = (const float4*)(xq + b * (16 * kLd) + 128 * g);
            const float4 x0 = p[0], x1 = p[1];
#pragma unroll
            for (int i = 0; i < kT; ++i) {
                const uint2 w8 = wv[b][i][g];
                const float sv = scale_s[i * (cols / 128) + k * kG + g];
                const wh_f2 w0 = wh_fp8x2<kSpecial, false>(w8.x), w1 = wh_fp8x2<kSpecial, true>(w8.x);
                const wh_f2 w2 = wh_fp8x2<kSpecial, false>(w8.y), w3 = wh_fp8x2<kSpecial, true>(w8.y);
                wh_f16 d;
#pragma unroll
                for (int r = 0; r < 16; ++r) d[r] = 0.0f;
                d = __builtin_amdgcn_mfma_f32_16x16x1f32(w0.x, x0.x, d, 0, 0, 0);
                d = __builtin_amdgcn_mfma_f32_16x16x1f32(w0.y, x0.y, d, 0, 0, 0);
                d = __builtin_amdgcn_mfma_f32_16x16x1f32(w1.x, x0.z, d, 0, 0, 0);
                d = __builtin_amdgcn_mfma_f32_16x16x1f32(w1.y, x0.w, d, 0, 0, 0);
                d = __builtin_amdgcn_mfma_f32_16x16x1f32(w2.x, x1.x, d, 0, 0, 0);
                d = __builtin_amdgcn_mfma_f32_16x16x1f32(w2.y, x1.y, d, 0, 0, 0);
                d = __builtin_amdgcn_mfma_f32_16x16x1f32(w3.x, x1.z, d, 0, 0, 0);
                d = __builtin_amdgcn_mfma_f32_16x16x1f32(w3.y, x1.w, d, 0, 0, 0);
                // block b's D[4 (lane / 16) + r][lane % 16] in d[4 b + r]
#pragma unroll
                for (int l = 0; l < 2; ++l)
#pragma unroll
                    for (int r = 0; r < 4; ++r)
                        acc[i][l][r] = __builtin_fmaf(d[8 * l + r] + d[8 * l + 4 + r], sv, acc[i][l][r]);
            }
        }
    };
    // chunk k in buffer k % 2; its weights and x are requested two chunks ahead
    // (the loop has no branch: where paths met, every load was waited for)
    load_x(0, 0);
    load_w(0, 0);
    load_x(1, 1);
    load_w(1, 1);
    store_x(0);
    __syncthreads();
    auto step = [&](uint32_t k, int b) {
        load_x(b, k + 2);
        __builtin_amdgcn_sched_barrier(0);
        chunk_mm(b, k);
        load_w(b, k + 2);
        __builtin_amdgcn_sched_barrier(0);
        store_x(b ^ 1);
        __syncthreads();
    };
    for (uint32_t k = 0; k < n_chunks; k += 2) {
        step(k, 0);
        step(k + 1, 1);
    }
    // the pairwise sum over l: l, l + 1 in the wave, the waves through LDS
    float* red = xs[0];  // [kT][4][16 inputs][17]
#pragma unroll
    for (int i = 0; i < kT; ++i)
#pragma unroll
        for (int r = 0; r < 4; ++r)
            red[((i * 4 + wave) * 16 + col) * 17 + 4 * q + r] = acc[i][0][r] + acc[i][1][r];
    __syncthreads();
    const uint32_t n = t >> 4, row = t & 15;
#pragma unroll
    for (int i = 0; i < kT; ++i) {
        const float* p = red + (i * 64 + n) * 17 + row;
        const float s = ((p[0] + p[16 * 17]) + (p[32 * 17] + p[48 * 17])) + 0.0f;
        const uint32_t out_row = row0 + 16 * i + row;
        if (n < n_here && out_row < r_hi) {
            yb[(size_t)(i0 + n) * a.y_stride + (out_row - r_lo)] = s;
            if (!(fabsf(s) <= 3.4028235e38f)) atomicOr(a.status, WH_ST_NONFINITE_OUTPUT);
        }
    }
}
