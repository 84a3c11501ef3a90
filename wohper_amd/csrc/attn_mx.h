// The window softmax of mla.h on f32 matrix instructions (gfx950), for the
// order-free numerics mode: the same keys, scores, weights, denominator and
// inverse RoPE (E/compute.rs:4106-4197) with the sums in another order.  Every
// product is an exact f32 FMA term of v_mfma_f32_16x16x4_f32, so no value is
// held or rounded in fewer bits than in the ordered kernels.
//
// Why: the ordered kernels add each score and output on one lane, two vector
// instructions a term, 80 % of their time.  64 heads x 628 keys of 32 positions are
// 2.6 GFLOP: 17 us at the 157 TFLOP/s of the f32 matrix rate, 128 us there.
//
// Two launches.  The scores of 32 keys leave as weights against that tile's
// own maximum, exp(score - tile max), with the maximum beside them; the second
// launch scales each tile by exp(tile max - max) as it reads it.  So the
// exponentials are made once and no launch only waits for a maximum.  A tile
// whose scores are all -inf counts against 0 (its weights are 0 once another
// tile is finite, and NaN when none is, as in the ordered kernels); NaN never
// wins a maximum.
#pragma once
#include "mla.h"

#define WH_ATTN_MX_KEYS 32u    // keys per score tile
#define WH_ATTN_MX_TILES 64u   // tiles per head at most (WH_ATTN_MAX_KEYS / 32)
#define WH_ATTN_MX_HEADS 256u  // heads at most: the tile maxima have a fixed room

struct wh_attn_f4 {  // four floats at any float's alignment
    float v[4];
} __attribute__((packed, aligned(4)));

// scores[h][j] = exp(q_h . key_j * scale - max of the tile) and tile_max.
// Grid (ceil(max_keys / 32), ceil(heads / 16), positions), 256 threads: wave w
// adds a quarter of the dims for 16 heads x 32 keys straight from global
// memory (a lane's 16 bytes are four dims of its row, the same four on both
// sides), LDS only joins the quarters.  For few positions, which 16 heads a
// workgroup leave enough workgroups; a batch takes k_attn_scores_mx_tile.
__global__ void __launch_bounds__(256) k_attn_scores_mx(wh_attn_args a) {
    constexpr int kS = 4;  // 16-dim steps requested together
    __shared__ __align__(16) float red[4][2][256];
    const wh_attn_pos v = wh_attn_resolve(a, blockIdx.z);
    const uint32_t t = threadIdx.x, wave = t >> 6, lane = t & 63, col = lane & 15, q = lane >> 4;
    const uint32_t nk = v.n_win + v.n_comp, hd = a.head_dim, n_s = hd / 64;
    const uint32_t j0 = blockIdx.x * WH_ATTN_MX_KEYS, h0 = blockIdx.y * 16;
    if (j0 >= nk) return;  // a batched launch's grid covers its longest key list
    const uint32_t base = wave * (hd / 4) + 4 * q;
    const float* const qp = v.q + (size_t)min(h0 + col, a.heads - 1) * hd + base;
    const float* kp[2];
#pragma unroll
    for (int k = 0; k < 2; ++k) kp[k] = wh_attn_key(a, v, min(j0 + 16 * k + col, nk - 1)) + base;
    wh_f4 qv[2][kS], kv[2][kS][2];
    auto request = [&](int b, uint32_t s0) {
#pragma unroll
        for (int s = 0; s < kS; ++s) {
            const uint32_t o = 16 * min(s0 + s, n_s - 1);
            qv[b][s] = *(const wh_f4*)(qp + o);
#pragma unroll
            for (int k = 0; k < 2; ++k) kv[b][s][k] = *(const wh_f4*)(kp[k] + o);
        }
    };
    wh_f4 acc[2];
    acc[0] = acc[1] = (wh_f4){0.0f, 0.0f, 0.0f, 0.0f};
    auto multiply = [&](int b, uint32_t s0) {
#pragma unroll
        for (int s = 0; s < kS; ++s) {
            if (s0 + s < n_s) {  // uniform
#pragma unroll
                for (int i = 0; i < 4; ++i)
#pragma unroll
                    for (int k = 0; k < 2; ++k)
                        acc[k] = __builtin_amdgcn_mfma_f32_16x16x4f32(qv[b][s][i], kv[b][s][k][i], acc[k], 0, 0, 0);
            }
        }
    };
    request(0, 0);
    for (uint32_t s0 = 0; s0 < n_s; s0 += 2 * kS) {
        request(1, s0 + kS);
        multiply(0, s0);
        if (s0 + 2 * kS < n_s) request(0, s0 + 2 * kS);
        multiply(1, s0 + kS);
    }
    // D[4 q + r][col]: head, key
#pragma unroll
    for (int k = 0; k < 2; ++k)
#pragma unroll
        for (int r = 0; r < 4; ++r) red[wave][k][(4 * q + r) * 16 + col] = acc[k][r];
    __syncthreads();
    // thread: two keys of one head, 16 threads a head
    const uint32_t e0 = (t & 15) * 2, h = h0 + (t >> 4);
    const uint32_t tile = e0 >> 4, at = (t >> 4) * 16 + (e0 & 15);
    const float ninf = -__uint_as_float(0x7f800000u);
    float s[2], mx = ninf;
#pragma unroll
    for (int e = 0; e < 2; ++e) {
        const float d = ((red[0][tile][at + e] + red[1][tile][at + e]) + (red[2][tile][at + e] + red[3][tile][at + e]));
        s[e] = d * a.scale;
        mx = fmaxf(mx, j0 + e0 + e < nk ? s[e] : ninf);
    }
#pragma unroll
    for (int off = 8; off >= 1; off >>= 1) mx = fmaxf(mx, __shfl_xor(mx, off, 64));
    const float ref = mx == ninf ? 0.0f : mx;
    if (h >= a.heads) return;
#pragma unroll
    for (int e = 0; e < 2; ++e) {
        const float w = wh_expf_glibc(s[e] - ref, kExpTab, kExpfExc, WH_EXPF_EXC_COUNT);
        if (j0 + e0 + e < nk) v.scores[(size_t)h * nk + j0 + e0 + e] = w;
    }
    if ((t & 15) == 0) a.tile_max[((size_t)blockIdx.z * a.heads + h) * WH_ATTN_MX_TILES + blockIdx.x] = mx;
}

// k_attn_scores_mx for a batch that fills the chip with 32 heads x 64 keys a
// workgroup: the queries and keys go through LDS 64 dims at a time, read in
// whole 256-byte pieces of their rows and requested two tiles ahead, and a
// wave takes 16 keys for all 32 heads, four sums a product (one per 16-dim
// step of a tile).  Read straight into the operands, every lane's 16 bytes
// were a row of their own, 64 cache lines an instruction, and a quarter of
// the dims a wave shared nothing.  64 heads x 628 keys of 32 positions:
// 40.5 -> 25.8 us (8.4 us of matrix time at 157 TFLOP/s).  The row stride of
// 68 floats puts the 16 rows of a read on 16 bank groups.
__global__ void __launch_bounds__(256) k_attn_scores_mx_tile(wh_attn_args a) {
    constexpr uint32_t kLd = 68;
    __shared__ __align__(16) float qs[2][32 * kLd], ks[2][64 * kLd];
    const wh_attn_pos v = wh_attn_resolve(a, blockIdx.z);
    const uint32_t t = threadIdx.x, wave = t >> 6, lane = t & 63, col = lane & 15, q = lane >> 4;
    const uint32_t nk = v.n_win + v.n_comp, hd = a.head_dim, n_t = hd / 64;
    const uint32_t j0 = blockIdx.x * 64, h0 = blockIdx.y * 32;
    if (j0 >= nk) return;  // a batched launch's grid covers its longest key list
    // staging: row t / 16 (+ 16 k), the 16-byte piece t % 16 of its 64 dims
    const float *qp[2], *kp[4];
    const uint32_t sr = t >> 4, sd = 4 * (t & 15);
#pragma unroll
    for (int k = 0; k < 2; ++k) qp[k] = v.q + (size_t)min(h0 + sr + 16 * k, a.heads - 1) * hd + sd;
#pragma unroll
    for (int k = 0; k < 4; ++k) kp[k] = wh_attn_key(a, v, min(j0 + sr + 16 * k, nk - 1)) + sd;
    wh_f4 qr[2][2], kr[2][4];
    auto request = [&](int b, uint32_t tile) {
        const uint32_t o = 64 * min(tile, n_t - 1);
#pragma unroll
        for (int k = 0; k < 2; ++k) qr[b][k] = *(const wh_f4*)(qp[k] + o);
#pragma unroll
        for (int k = 0; k < 4; ++k) kr[b][k] = *(const wh_f4*)(kp[k] + o);
    };
    auto store = [&](int b) {
#pragma unroll
        for (int k = 0; k < 2; ++k) *(wh_f4*)(qs[b] + (sr + 16 * k) * kLd + sd) = qr[b][k];
#pragma unroll
        for (int k = 0; k < 4; ++k) *(wh_f4*)(ks[b] + (sr + 16 * k) * kLd + sd) = kr[b][k];
    };
    wh_f4 acc[4][2];
#pragma unroll
    for (int s = 0; s < 4; ++s) acc[s][0] = acc[s][1] = (wh_f4){0.0f, 0.0f, 0.0f, 0.0f};
    auto multiply = [&](int b) {
        const float* qb = qs[b] + col * kLd + 4 * q;
        const float* kb = ks[b] + (16 * wave + col) * kLd + 4 * q;
#pragma unroll
        for (int s = 0; s < 4; ++s) {
            const wh_f4 q0 = *(const wh_f4*)(qb + 16 * s), q1 = *(const wh_f4*)(qb + 16 * kLd + 16 * s);
            const wh_f4 k = *(const wh_f4*)(kb + 16 * s);
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                acc[s][0] = __builtin_amdgcn_mfma_f32_16x16x4f32(q0[i], k[i], acc[s][0], 0, 0, 0);
                acc[s][1] = __builtin_amdgcn_mfma_f32_16x16x4f32(q1[i], k[i], acc[s][1], 0, 0, 0);
            }
        }
    };
    // tile k in buffer k % 2
    request(0, 0);
    request(1, 1);
    store(0);
    __syncthreads();
    auto step = [&](uint32_t k, int b) {
        request(b, k + 2);
        multiply(b);
        store(b ^ 1);
        __syncthreads();
    };
    // no branch inside the loop: where paths met, every load was waited for
    for (uint32_t k = 0; k + 2 <= n_t; k += 2) {
        step(k, 0);
        step(k + 1, 1);
    }
    if (n_t & 1) step(n_t - 1, 0);
    float* sc = ks[0];  // [32 heads][64 keys]
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int r = 0; r < 4; ++r)
            sc[(16 * h + 4 * q + r) * kLd + 16 * wave + col] = (acc[0][h][r] + acc[1][h][r]) + (acc[2][h][r] + acc[3][h][r]);
    __syncthreads();
    // thread: eight keys of one head, four threads a 32-key tile
    const uint32_t hl = t >> 3, e0 = (t & 7) * 8, h = h0 + hl;
    const float ninf = -__uint_as_float(0x7f800000u);
    float s[8], mx = ninf;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
        s[e] = sc[hl * kLd + e0 + e] * a.scale;
        mx = fmaxf(mx, j0 + e0 + e < nk ? s[e] : ninf);
    }
    mx = fmaxf(mx, wh_dpp_f<0xB1>(mx));
    mx = fmaxf(mx, wh_dpp_f<0x4E>(mx));
    const float ref = mx == ninf ? 0.0f : mx;
    if (h >= a.heads) return;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
        const float w = wh_expf_glibc(s[e] - ref, kExpTab, kExpfExc, WH_EXPF_EXC_COUNT);
        if (j0 + e0 + e < nk) v.scores[(size_t)h * nk + j0 + e0 + e] = w;
    }
    const uint32_t tile = 2 * blockIdx.x + (e0 >> 5);
    if ((t & 3) == 0 && tile * WH_ATTN_MX_KEYS < nk)
        a.tile_max[((size_t)blockIdx.z * a.heads + h) * WH_ATTN_MX_TILES + tile] = mx;
}

// out = (sum of weights x keys) / denominator, then the inverse RoPE.  Grid
// (head_dim / (16 kD), ceil(heads / (16 kH)), positions), 256 threads: the
// waves take every fourth 16 keys, LDS joins them.
template <int kH, int kD>
__global__ void __launch_bounds__(256) k_attn_weighted_mx(wh_attn_args a) {
    __shared__ __align__(16) float red[4][kH * kD][256];
    __shared__ float den_s[4][16 * kH], max_s[16 * kH];
    __shared__ float f_s[16 * kH][WH_ATTN_MX_TILES + 1];  // exp(tile max - max)
    const wh_attn_pos v = wh_attn_resolve(a, blockIdx.z);
    const uint32_t t = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(t >> 6), lane = t & 63, col = lane & 15, q = lane >> 4;
    const uint32_t nk = v.n_win + v.n_comp, hd = a.head_dim;
    const uint32_t d0 = blockIdx.x * (16 * kD), h0 = blockIdx.y * (16 * kH);
    const uint32_t nt = (nk + WH_ATTN_MX_KEYS - 1) / WH_ATTN_MX_KEYS, n_full = nk / 16;
    const float* wrow[kH];
#pragma unroll
    for (int h = 0; h < kH; ++h) wrow[h] = v.scores + (size_t)min(h0 + 16 * h + col, a.heads - 1) * nk;
    float w[2][kH][4], x[2][4][kD];
    // 16 keys from 16 u: lane q the keys 4 q .. + 3 of its head and of its dims.
    // Whole units only, always as many loads and no branch, so that two units
    // stay in flight (with a branch for a partial one every product waited for
    // every load: one position over 1128 keys 18.3 us then, 16.0 us so, both
    // launches); a last partial unit comes after the loop
    auto request = [&](int b, uint32_t u) {
        const uint32_t j = 16 * min(u, n_full - 1) + 4 * q;
#pragma unroll
        for (int h = 0; h < kH; ++h) {
            const wh_attn_f4 p = *(const wh_attn_f4*)(wrow[h] + j);
#pragma unroll
            for (int i = 0; i < 4; ++i) w[b][h][i] = p.v[i];
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const float* row = wh_attn_key(a, v, j + i) + d0 + col;
#pragma unroll
            for (int c = 0; c < kD; ++c) x[b][i][c] = row[16 * c];
        }
    };
    if (n_full) {  // uniform
        request(0, wave);
        request(1, wave + 4);
    }
    // the heads' maxima and their tiles' factors: 16 threads a head
#pragma unroll
    for (int h = 0; h < kH; ++h) {
        const uint32_t hl = 16 * h + (t >> 4);
        const float* tm = a.tile_max + ((size_t)blockIdx.z * a.heads + min(h0 + hl, a.heads - 1)) * WH_ATTN_MX_TILES;
        const float ninf = -__uint_as_float(0x7f800000u);
        float m[WH_ATTN_MX_TILES / 16], mx = ninf;
#pragma unroll
        for (int k = 0; k < (int)WH_ATTN_MX_TILES / 16; ++k) {
            const uint32_t tile = (t & 15) + 16 * k;
            m[k] = tile < nt ? tm[tile] : ninf;
            mx = fmaxf(mx, m[k]);
        }
#pragma unroll
        for (int off = 8; off >= 1; off >>= 1) mx = fmaxf(mx, __shfl_xor(mx, off, 64));
#pragma unroll
        for (int k = 0; k < (int)WH_ATTN_MX_TILES / 16; ++k)
            if (16 * k < nt) f_s[hl][(t & 15) + 16 * k] = wh_expf_glibc(m[k] - mx, kExpTab, kExpfExc, WH_EXPF_EXC_COUNT);
        if ((t & 15) == 0) max_s[hl] = mx;
    }
    __syncthreads();
    wh_f4 acc[kH][kD];
    float den[kH];
#pragma unroll
    for (int h = 0; h < kH; ++h) {
        den[h] = 0.0f;
#pragma unroll
        for (int c = 0; c < kD; ++c) acc[h][c] = (wh_f4){0.0f, 0.0f, 0.0f, 0.0f};
    }
    auto multiply = [&](int b, uint32_t u) {
#pragma unroll
        for (int h = 0; h < kH; ++h) {
            const float f = f_s[16 * h + col][u >> 1];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const float p = w[b][h][i] * f;
                den[h] = den[h] + p;
#pragma unroll
                for (int c = 0; c < kD; ++c)
                    acc[h][c] = __builtin_amdgcn_mfma_f32_16x16x4f32(p, x[b][i][c], acc[h][c], 0, 0, 0);
            }
        }
    };
    for (uint32_t u = wave; u < n_full; u += 8) {
        multiply(0, u);
        request(0, u + 8);
        if (u + 4 < n_full) multiply(1, u + 4);  // uniform, and no loads in it
        request(1, u + 12);
    }
    if (nk % 16 && wave == (n_full & 3)) {  // uniform: the wave with the fewest units
        const uint32_t j = 16 * n_full + 4 * q;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const bool on = j + i < nk;
            const uint32_t jc = on ? j + i : nk - 1;
            const float* row = wh_attn_key(a, v, jc) + d0 + col;
#pragma unroll
            for (int c = 0; c < kD; ++c) {
                const float xv = row[16 * c];
                x[0][i][c] = on ? xv : 0.0f;
            }
#pragma unroll
            for (int h = 0; h < kH; ++h) {
                const float wv = wrow[h][jc];
                w[0][h][i] = on ? wv : 0.0f;
            }
        }
        multiply(0, n_full);
    }
#pragma unroll
    for (int h = 0; h < kH; ++h) {
        den[h] = den[h] + __shfl_xor(den[h], 16, 64);
        den[h] = den[h] + __shfl_xor(den[h], 32, 64);
        if (q == 0) den_s[wave][16 * h + col] = den[h];
#pragma unroll
        for (int c = 0; c < kD; ++c)
#pragma unroll
            for (int r = 0; r < 4; ++r) red[wave][h * kD + c][(4 * q + r) * 16 + col] = acc[h][c][r];
    }
    __syncthreads();
    // thread: dim t % 16 of every tile's head t / 16
#pragma unroll
    for (int c = 0; c < kD; ++c) {
        const uint32_t d = d0 + 16 * c + (t & 15), p = (d - a.nope_dim) / 2;
        const bool any = d0 + 16 * c + 15 >= a.nope_dim && d0 + 16 * c < a.nope_dim + 2 * a.pairs;  // uniform
        const bool on = any && d >= a.nope_dim && p < a.pairs;
        float sn = 0.0f, cs = 1.0f;
        if (any) {
            const float ang = (float)v.token_pos * (on ? a.inv_freqs[p] : 0.0f);
            sn = -wh_sincosf_glibc(ang, 0);
            cs = wh_sincosf_glibc(ang, 1);
        }
#pragma unroll
        for (int h = 0; h < kH; ++h) {
            const uint32_t hl = 16 * h + (t >> 4), hh = h0 + hl;
            float y = (red[0][h * kD + c][t] + red[1][h * kD + c][t]) + (red[2][h * kD + c][t] + red[3][h * kD + c][t]);
            float dn = (den_s[0][hl] + den_s[1][hl]) + (den_s[2][hl] + den_s[3][hl]);
            if (a.sink)
                dn = wh_expf_glibc(a.sink[min(hh, a.heads - 1)] - max_s[hl], kExpTab, kExpfExc, WH_EXPF_EXC_COUNT) + dn;
            if (dn > 0.0f) y = y / dn;
            if (any) {
                const float other = __shfl_xor(y, 1, 64);
                if (on) y = (d & 1) ? other * sn + y * cs : y * cs - other * sn;
            }
            if (hh < a.heads) v.out[(size_t)hh * hd + d] = y;
        }
    }
}
