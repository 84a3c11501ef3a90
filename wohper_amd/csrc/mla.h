// The non-GEMV glue of a DeepSeek-V4 MLA attention layer at decode, on
// gfx950: RMS norms, interleaved RoPE / YaRN, the act-quant between
// projections, and the sliding-window softmax with attention sink
// (compute_deepseek_v4_mla_attention, E/compute.rs:3924-4293).
//
// Every value follows the reference's f32 arithmetic bit for bit: sums run
// in the reference's sequential order (one lane per chain), products and
// sums are separate roundings (the library is built without contraction),
// exp / sin / cos are the glibc-exact restatements of libm_emul.h, and the
// act-quant is the block-64 rule of E/compute.rs:2504-2521.  The data are a
// few hundred KB per token, so these kernels are latency-bound: they keep
// the hidden state on the device between the FP8 projections rather than
// aiming at bandwidth.
#pragma once
#include "kernels.h"

#define WH_ROWPOST_MAX 4096u     // values per row of k_rowpost
#define WH_ATTN_MAX_KEYS 2048u   // window + compressed keys per head
#define WH_ATTN_MAX_HEAD_DIM 1024u
#define WH_POS_BATCH 128u        // positions per batched launch of k_rowpost / the attention

__device__ __forceinline__ float wh_bf16_value(uint16_t raw) { return __uint_as_float((uint32_t)raw << 16); }

// Act-quant (E/compute.rs:2504-2521) of one 64-value block held one value
// per lane of a wave; lanes past the block's end pass valid = false (they
// add nothing to the block maximum, as the reference's shorter tail chunk).
__device__ __forceinline__ float wh_aq64_wave(float x, bool valid) {
    float amax = wh_wave_max(valid ? fabsf(x) : 0.0f);
    amax = fmaxf(amax, 1.0e-4f);
    const bool inf_scale = !(amax <= 3.4028235e38f);
    const int k = inf_scale ? 0 : wh_aq_scale_exp(amax, kLog2Thr);
    const float scale = inf_scale ? __uint_as_float(0x7f800000u) : wh_pow2f(k);
    const float inv = inf_scale ? 0.0f : wh_pow2f(-k);
    const float t = inf_scale ? x / scale : x * inv;
    const float q = t != t ? -480.0f : wh_e4m3_round(wh_clamp448(t));  // NaN -> the lowest LUT entry
    return q * scale;
}

// ------------------------------------------------------------- row glue
// Per row r (one workgroup of 256 threads each), in this order, on
// x + r * ld_in, n values:
//   norm:  rms_norm_in_place (E/compute.rs:7110-7122) when w is null, else
//          apply_weighted_rms_norm (E/compute.rs:3077-3107) with bf16 w:
//          s = sequential sum of v*v, inv = 1 / sqrt(s / n + 1e-6),
//          v = v * inv (* w);
//   rope:  apply_rope_interleaved_with_freqs (E/compute.rs:2623-2649) on
//          [rope_off, rope_off + 2 pairs) at `position`, inverse or not;
//   quant: act-quant, block 64, of [0, aq_len);
// then the row goes to out + r * ld_out (which may be x).
struct wh_rowpost_args {
    const float* x;
    float* out;
    uint32_t rows, n, ld_in, ld_out;
    uint32_t norm;              // 0: no norm
    const uint16_t* w;          // bf16 [n] or null
    const float* inv_freqs;     // [pairs]
    uint32_t pairs, rope_off, position, inverse;
    uint32_t aq_len;            // 0: no act-quant
    uint32_t tree;              // norm: 1 = the sum of squares in a fixed tree (exact numerics off)
    // several positions in one launch: rows_per_pos > 0 puts row r at
    // position bpos[r / rows_per_pos] (in place of `position`); out_at_pos
    // sends row r to out + bpos[r] * ld_out (one row per position: a KV
    // cache row)
    uint32_t rows_per_pos, out_at_pos;
    uint32_t bpos[WH_POS_BATCH];
    // hc > 0: the row is the end of hc_pre_into (E/compute.rs:5044-5050),
    // y[d] = sum over i in order of hc_pre[r * hc + i] * x[i * hc_stride + d]
    // for the hc copies at x + r * ld_in, instead of x itself
    const float* hc_pre;
    uint32_t hc, hc_stride;
};

// One row by kT threads (256, or 1024 for a lone row); each thread's values
// and norm weights are loaded up front.
template <int kT>
__device__ __forceinline__ void wh_rowpost_row(const wh_rowpost_args& a, uint32_t row) {
    constexpr int kPer = WH_ROWPOST_MAX / kT;  // values per thread at most
    constexpr int kW = kT / 64;                // waves
    __shared__ __align__(16) float v[WH_ROWPOST_MAX];
    __shared__ float inv_s;
    const uint32_t t = threadIdx.x, n = a.n;
    const float* x = a.x + (size_t)row * a.ld_in;
    uint32_t position = a.position;
    size_t orow = row;
    if (a.rows_per_pos) {
        position = a.bpos[row / a.rows_per_pos];
        if (a.out_at_pos) orow = position;
    }
    float xv[kPer], wv[kPer];
    // every load issued before any is used, from clamped indices (a load
    // under a branch is waited for on its own; with no norm weights the
    // row itself stands in as a valid address)
    const bool use_w = a.norm && a.w;
    const uint16_t* wp = use_w ? a.w : (const uint16_t*)x;
    uint32_t wr[kPer];
    if (a.hc == 4) {
        // the four copies' loads issued together, then the reference's sum
        const float* pre = a.hc_pre + (size_t)row * 4;
        const float p0 = pre[0], p1 = pre[1], p2 = pre[2], p3 = pre[3];
        float cv[4][kPer];
#pragma unroll
        for (int k = 0; k < kPer; ++k) {
            const uint32_t i = t + kT * k, ic = i < n ? i : 0u;
#pragma unroll
            for (int j = 0; j < 4; ++j) cv[j][k] = x[(size_t)j * a.hc_stride + ic];
            wr[k] = wp[ic];
        }
#pragma unroll
        for (int k = 0; k < kPer; ++k) {
            float acc = 0.0f;
            acc = acc + p0 * cv[0][k];
            acc = acc + p1 * cv[1][k];
            acc = acc + p2 * cv[2][k];
            acc = acc + p3 * cv[3][k];
            xv[k] = acc;
        }
    } else if (a.hc) {
        const float* pre = a.hc_pre + (size_t)row * a.hc;
#pragma unroll
        for (int k = 0; k < kPer; ++k) {
            const uint32_t i = t + kT * k, ic = i < n ? i : 0u;
            float acc = 0.0f;
            for (uint32_t j = 0; j < a.hc; ++j) acc = acc + pre[j] * x[(size_t)j * a.hc_stride + ic];
            xv[k] = acc;
            wr[k] = wp[ic];
        }
    } else {
#pragma unroll
        for (int k = 0; k < kPer; ++k) {
            const uint32_t i = t + kT * k, ic = i < n ? i : 0u;
            xv[k] = x[ic];
            wr[k] = wp[ic];
        }
    }
#pragma unroll
    for (int k = 0; k < kPer; ++k) {
        const uint32_t i = t + kT * k;
        if (i >= n) xv[k] = 0.0f;
        wv[k] = use_w && i < n ? wh_bf16_value((uint16_t)wr[k]) : 1.0f;
    }
    if (!a.norm) {
#pragma unroll
        for (int k = 0; k < kPer; ++k)
            if (t + kT * k < n) v[t + kT * k] = xv[k];
        __syncthreads();
    } else {
        if (a.tree) {
            // each thread its strided terms, then the wave butterfly, then
            // the waves in order: the same value up to rounding
            __shared__ float red[kW];
            float s = 0.0f;
#pragma unroll
            for (int k = 0; k < kPer; ++k) s = s + xv[k] * xv[k];  // zeros past n
            for (int off = 32; off > 0; off >>= 1) s = s + __shfl_xor(s, off, 64);
            if ((t & 63) == 0) red[t >> 6] = s;
            __syncthreads();
            if (t == 0) {
                float r = red[0];
#pragma unroll
                for (int w = 1; w < kW; ++w) r = r + red[w];
                inv_s = 1.0f / sqrtf(r / (float)n + 1.0e-6f);
            }
        } else {
            // the reference's order: every product rounded on its own, then
            // the sequential sum by the whole workgroup (ordered_sum.h); up
            // to 576 terms one lane adds them (one row of 513 4.0 us that
            // way and 4.6 with the tables and the check, of 600 5.1 and 4.6)
            constexpr int kMaxL = WH_ROWPOST_MAX / 32;
            __shared__ __align__(16) wh_osum_lds<kMaxL, 32> os;
            auto stage = [&](auto l) {
                constexpr int kL = decltype(l)::value;
                auto& s = *(wh_osum_lds<kL, 32>*)&os;
#pragma unroll
                for (int k = 0; k < kPer; ++k) {
                    const uint32_t i = t + kT * k;
                    if (i < 32 * kL) s.rows[wh_osum_at<kL>(i)] = i < n ? xv[k] * xv[k] : -0.0f;
                }
                return wh_ordered_sum_wg<kT, kL, 32>(s, 0.0f);
            };
            float s;
            if (n <= 576) {
#pragma unroll
                for (int k = 0; k < (576 + kT - 1) / kT; ++k)
                    if (t + kT * k < n) os.rows[t + kT * k] = xv[k] * xv[k];
                __syncthreads();
                s = t == 0 ? wh_ordered_sum_lds(os.rows, n, 0.0f) : 0.0f;
            } else if (n <= 1024) {
                s = stage(std::integral_constant<int, 32>());
            } else if (n <= 2048) {
                s = stage(std::integral_constant<int, 64>());
            } else {
                s = stage(std::integral_constant<int, kMaxL>());
            }
            if (t == 0) inv_s = 1.0f / sqrtf(s / (float)n + 1.0e-6f);
        }
        __syncthreads();
        const float inv = inv_s;
#pragma unroll
        for (int k = 0; k < kPer; ++k) {
            const uint32_t i = t + kT * k;
            if (i < n) {
                float y = xv[k] * inv;
                if (a.w) y = y * wv[k];
                v[i] = y;
            }
        }
        __syncthreads();
    }
    if (a.pairs) {
        const float pos = (float)position;
        for (uint32_t p = t; p < a.pairs; p += kT) {
            const float ang = pos * a.inv_freqs[p];
            float sn = wh_sincosf_glibc(ang, 0);
            const float cs = wh_sincosf_glibc(ang, 1);
            if (a.inverse) sn = -sn;
            float* pv = v + a.rope_off + 2 * p;
            const float e = pv[0], o = pv[1];
            pv[0] = e * cs - o * sn;
            pv[1] = e * sn + o * cs;
        }
        __syncthreads();
    }
    if (a.aq_len && a.aq_len % 64 == 0) {
        // whole blocks: 16 lanes each, every thread a quarter of the steps a
        // value per lane takes (4096 values by 256 threads: the row kernel
        // 15.8 -> 10.4 us for 128 rows, 13.6 -> 7.1 us for 32)
        for (uint32_t i = 4 * t; i < a.aq_len; i += 4 * kT) {
            float4* const p = (float4*)(v + i);
            *p = wh_aq64_quad(*p);
        }
        __syncthreads();
    } else if (a.aq_len) {
        const uint32_t wave = t >> 6, lane = t & 63;
        for (uint32_t b = wave; b * 64 < a.aq_len; b += kW) {
            const uint32_t i = b * 64 + lane;
            const bool valid = i < a.aq_len;
            const float q = wh_aq64_wave(valid ? v[i] : 0.0f, valid);
            if (valid) v[i] = q;
        }
        __syncthreads();
    }
    float* out = a.out + orow * a.ld_out;
    for (uint32_t i = t; i < n; i += kT) out[i] = v[i];
}

template <int kT>
__global__ void __launch_bounds__(kT) k_rowpost(wh_rowpost_args a) {
    wh_rowpost_row<kT>(a, blockIdx.x);
}

// Two row sets that do not depend on each other in one launch: the low-rank
// q's norm and the cache rows of a position, each a launch of a few
// workgroups bound by its chain of barriers (4 to 7 us).
struct wh_rowpost_pair {
    wh_rowpost_args r[2];
};
template <int kT>
__global__ void __launch_bounds__(kT) k_rowpost_pair(wh_rowpost_pair p) {
    const uint32_t first = p.r[0].rows, second = blockIdx.x >= first ? 1u : 0u;
    wh_rowpost_row<kT>(p.r[second], blockIdx.x - (second ? first : 0u));
}

// k_rowpost for rows of 512 with the norm (no weights, the sum in the fixed
// tree) and RoPE only: the heads of q with exact numerics off.  One wave a
// row, no LDS and no barrier: lane L holds elements 64 k + L, so the tree's
// four waves are four butterflies of this one and a rotated pair sits in
// neighbouring lanes.  The same bits.  Bound by memory: 8192 heads, 33.6 MB
// both ways, 11.0 us; with a workgroup a row, five barriers and a 16 KB
// copy of it in LDS, 37.4 us (in four launches).  blockDim / 64 rows a workgroup.
__global__ void __launch_bounds__(256) k_rowpost_heads(wh_rowpost_args a) {
    const uint32_t lane = threadIdx.x & 63, row = blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6);
    if (row >= a.rows) return;  // a whole wave
    const float* x = a.x + (size_t)row * a.ld_in + lane;
    float xv[8];
#pragma unroll
    for (int k = 0; k < 8; ++k) xv[k] = x[64 * k];
    float s[4];
#pragma unroll
    for (int w = 0; w < 4; ++w) s[w] = (0.0f + xv[w] * xv[w]) + xv[w + 4] * xv[w + 4];
    for (int off = 32; off > 0; off >>= 1)
#pragma unroll
        for (int w = 0; w < 4; ++w) s[w] = s[w] + __shfl_xor(s[w], off, 64);
    const float inv = 1.0f / sqrtf((((s[0] + s[1]) + s[2]) + s[3]) / 512.0f + 1.0e-6f);
    const float pos = (float)(a.rows_per_pos ? a.bpos[row / a.rows_per_pos] : a.position);
    float* out = a.out + (size_t)row * a.ld_out + lane;
#pragma unroll
    for (int k = 0; k < 8; ++k) {
        float y = xv[k] * inv;
        if (64u * k + 63 >= a.rope_off && 64u * k < a.rope_off + 2 * a.pairs) {  // uniform
            const uint32_t i = 64 * k + lane, p = (i - a.rope_off) >> 1;
            const bool on = i >= a.rope_off && p < a.pairs;
            const float ang = pos * (on ? a.inv_freqs[p] : 0.0f);
            float sn = wh_sincosf_glibc(ang, 0);
            const float cs = wh_sincosf_glibc(ang, 1);
            if (a.inverse) sn = -sn;
            const float other = __shfl_xor(y, 1, 64);
            if (on) y = (i & 1) ? other * sn + y * cs : y * cs - other * sn;
        }
        out[64 * k] = y;
    }
}

// --------------------------------------------------------- window softmax
// Keys of one decode position: the window rows (the KV cache at positions
// [window_start, token_pos], row stride win_ld) then the visible compressed
// rows (head_dim apart), E/compute.rs:4106-4160.
struct wh_attn_args {
    const float* q;        // [heads][head_dim]
    const float* win;      // first window row
    const float* comp;     // compressed rows
    const float* sink;     // [heads] or null
    const float* inv_freqs;
    float* scores;         // [heads][n_keys] scratch
    float* out;            // [heads][head_dim]
    uint32_t heads, head_dim, nope_dim, pairs;
    uint32_t n_win, n_comp, win_ld, token_pos;
    float scale;           // head_dim^-0.5 (host powf, as the reference)
    // a batch of positions (nb > 0): slot z takes q and out +
    // z * q_ld, scores + z * scores_ld, token_pos = bpos[z], the window of
    // the last wlen cache rows up to that position (win = the cache's row
    // 0), compressed rows bcomp[z] (bncomp[z] of them)
    uint32_t nb, q_ld, scores_ld, wlen;
    uint32_t max_keys;     // the longest key list
    float* tile_max;       // attn_mx.h: [nb][heads][64]
    uint32_t wts_ld;       // k_attn_combine: floats per head of its dynamic LDS (>= every n_keys)
    uint32_t bpos[WH_POS_BATCH];
    uint32_t bncomp[WH_POS_BATCH];
    const float* bcomp[WH_POS_BATCH];
};

// One position's keys, queries and outputs.
struct wh_attn_pos {
    const float* q;
    const float* win;
    const float* comp;
    float* scores;
    float* out;
    uint32_t n_win, n_comp, token_pos;
};

__device__ __forceinline__ wh_attn_pos wh_attn_resolve(const wh_attn_args& a, uint32_t z) {
    wh_attn_pos v{a.q, a.win, a.comp, a.scores, a.out, a.n_win, a.n_comp, a.token_pos};
    if (a.nb) {
        const uint32_t p = a.bpos[z], context = p + 1;
        const uint32_t ws = context > a.wlen ? context - a.wlen : 0u;
        v.q = a.q + (size_t)z * a.q_ld;
        v.out = a.out + (size_t)z * a.q_ld;
        v.scores = a.scores + (size_t)z * a.scores_ld;
        v.win = a.win + (size_t)ws * a.win_ld;
        v.n_win = context - ws;
        v.comp = a.bcomp[z];
        v.n_comp = a.bncomp[z];
        v.token_pos = p;
    }
    return v;
}

__device__ __forceinline__ const float* wh_attn_key(const wh_attn_args& a, const wh_attn_pos& v, uint32_t j) {
    return j < v.n_win ? v.win + (size_t)j * a.win_ld : v.comp + (size_t)(j - v.n_win) * a.head_dim;
}

// v(lane kI of each row of 16 lanes) * x: a DPP row broadcast is part of the
// multiplication, so sixteen uniform factors in one register, the same in
// every row, cost no instruction of their own.
template <int kI>
__device__ __forceinline__ float wh_mul_bcast(float v, float x) {
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x150 + kI, 0xf, 0xf, true)) * x;
}

// scores[h][j] = (sum over d, in order, of q[h][d] * key_j[d]) * scale.
// Grid (ceil(n_keys / 64), ceil(heads / (4 kR)), positions), 256 threads: a
// lane takes one key, a wave kR heads: two vector instructions per dim, head
// and wave, which is what bounds a batch (q through scalar loads or readlane
// was slower: 78 and 61 against 51 us for 64 heads x 628 keys of 32
// positions, 80% of it vector issue; before, four heads a workgroup and both
// factors of every product from LDS, 107 us).  The workgroup's 64 keys go through LDS 64 dims at a
// time, two tiles in turn (one barrier a tile; row stride 68 floats: the
// lanes' 16-byte reads fall in distinct banks), requested 8 (four heads
// a wave: 4) tiles at a time so that the launch waits for one memory round
// trip; the next dims' reads
// are in flight while the current ones are added.  More heads per wave read
// a key fewer times and leave fewer waves: see attn_launch.
#define WH_ATTN_TILE_LD 68u  // floats per key of a score tile
template <int kR>
__global__ void __launch_bounds__(256) k_attn_scores(wh_attn_args a) {
    constexpr int kPre = kR == 4 ? 4 : 8;  // tiles requested together
    __shared__ __align__(16) float tile[2][64 * WH_ATTN_TILE_LD];
    const wh_attn_pos v = wh_attn_resolve(a, blockIdx.z);
    const uint32_t t = threadIdx.x, wave = t >> 6, lane = t & 63;
    const uint32_t h0 = (blockIdx.y * 4 + wave) * kR, j0 = blockIdx.x * 64;
    const uint32_t nk = v.n_win + v.n_comp, hd = a.head_dim, n_ch = hd / 64;
    if (j0 >= nk) return;  // a batched launch's grid covers its longest key list
    // staging: thread t copies float4 t % 16 of keys t / 16 + 16 i of a tile
    const uint32_t kk = t >> 4, f4 = t & 15;
    const float* krow[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const uint32_t j = j0 + kk + 16 * i;
        krow[i] = wh_attn_key(a, v, j < nk ? j : j0) + 4 * f4;  // keys past the end: not stored
    }
    wh_f4 kv[kPre][4];
    float qv[kPre][kR][4];  // of 16 dims each: lane i dim i % 16
    auto request = [&](uint32_t c0) {
#pragma unroll
        for (int c = 0; c < kPre; ++c) {
            const uint32_t cc = c0 + c < n_ch ? c0 + c : 0u;
#pragma unroll
            for (int i = 0; i < 4; ++i) kv[c][i] = *(const wh_f4*)(krow[i] + 64 * cc);
#pragma unroll
            for (int r = 0; r < kR; ++r)
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    qv[c][r][i] = v.q[(size_t)(h0 + r < a.heads ? h0 + r : a.heads - 1) * hd + 64 * cc + 16 * i +
                                      (lane & 15)];
        }
    };
    request(0);
    constexpr int kS = 16;  // dims per stage
    float s[kR];
#pragma unroll
    for (int r = 0; r < kR; ++r) s[r] = 0.0f;
    for (uint32_t c0 = 0; c0 < n_ch; c0 += kPre) {
        if (c0) request(c0);
        wh_static_for<kPre>([&](auto cc) {
            constexpr int c = decltype(cc)::value;
            if (c0 + c < n_ch) {  // uniform
                float* dst = tile[c & 1];
#pragma unroll
                for (int i = 0; i < 4; ++i) *(wh_f4*)(dst + (kk + 16 * i) * WH_ATTN_TILE_LD + 4 * f4) = kv[c][i];
                __syncthreads();  // and the reads of the tile before this one's last use are done
                const float* src = tile[c & 1] + lane * WH_ATTN_TILE_LD;
                wh_f4 kr[2][kS / 4];
                auto read = [&](int b, int st) {
#pragma unroll
                    for (int i = 0; i < kS / 4; ++i) kr[b][i] = *(const wh_f4*)(src + kS * st + 4 * i);
                };
                read(0, 0);
#pragma unroll
                for (int st = 0; st < 64 / kS; ++st) {
                    if (st + 1 < 64 / kS) read((st + 1) & 1, st + 1);
                    __builtin_amdgcn_sched_barrier(0);
                    wh_static_for<kS>([&](auto ii) {
                        constexpr int i = decltype(ii)::value;
                        const float k = kr[st & 1][i >> 2][i & 3];
#pragma unroll
                        for (int r = 0; r < kR; ++r) s[r] = s[r] + wh_mul_bcast<i>(qv[c][r][st], k);
                    });
                    __builtin_amdgcn_sched_barrier(0);
                }
            }
        });
    }
    const uint32_t j = j0 + lane;
#pragma unroll
    for (int r = 0; r < kR; ++r)
        if (h0 + r < a.heads && j < nk) v.scores[(size_t)(h0 + r) * nk + j] = s[r] * a.scale;
}

// The keys' 64 dims d0 .. d0 + 63 of a workgroup through LDS, 64 keys a tile,
// two tiles in turn, four requested ahead.
struct wh_attn_tiles {
    wh_f4 kv[4][4];
    uint32_t kk, f4;  // thread t copies float4 t % 16 of keys t / 16 + 16 i
    __device__ __forceinline__ void request(const wh_attn_args& a, const wh_attn_pos& v, uint32_t nk, uint32_t j0,
                                            wh_f4 (&r)[4]) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const uint32_t j = j0 + kk + 16 * i;  // past the last key: key 0's bytes, never used
            r[i] = *(const wh_f4*)(wh_attn_key(a, v, j < nk ? j : 0u) + blockIdx.x * 64 + 4 * f4);
        }
    }
    // per tile, all threads: ahead(j0) for its keys' other loads, then
    // body(tile, j0, keys).  Tiles come in fours and are requested whether
    // they hold keys or not: with no load under a branch the compiler's waits
    // cover exactly the tile that is stored (a load it cannot count makes
    // every wait one for all loads, 1.3 us a tile).
    template <class Ahead, class Body>
    __device__ __forceinline__ void run(const wh_attn_args& a, const wh_attn_pos& v, uint32_t nk,
                                        float (*tile)[64 * 64], Ahead ahead, Body body) {
        for (uint32_t j0 = 0; j0 < nk; j0 += 256) {
            wh_static_for<4>([&](auto ii) {
                constexpr int i = decltype(ii)::value;
                float* dst = tile[i & 1];
#pragma unroll
                for (int k = 0; k < 4; ++k) *(wh_f4*)(dst + (kk + 16 * k) * 64 + 4 * f4) = kv[i][k];
                ahead(ii, j0 + 64 * i);
                request(a, v, nk, j0 + 64 * i + 256, kv[i]);
                __syncthreads();  // and the reads of the tile before this one's last use are done
                if (j0 + 64 * i < nk) body(ii, (const float*)tile[i & 1], j0 + 64 * i, min(64u, nk - (j0 + 64 * i)));
            });
        }
    }
    __device__ __forceinline__ void start(const wh_attn_args& a, const wh_attn_pos& v, uint32_t nk) {
        kk = threadIdx.x >> 4;
        f4 = threadIdx.x & 15;
#pragma unroll
        for (uint32_t i = 0; i < 4; ++i) request(a, v, nk, 64 * i, kv[i]);
    }
};

// f(sixteen b, key i, key's value) for keys 16 b + i < m of a tile, in order;
// tp: the lane's dim of the tile's key 0.  A full tile is straight-line code
// with the next sixteen keys' reads in flight.
template <class F>
__device__ __forceinline__ void wh_attn_keys(const float* tp, uint32_t m, F f) {
    float x[2][16];
    auto read = [&](int s, int b) {
#pragma unroll
        for (int i = 0; i < 16; ++i) x[s][i] = tp[64 * (16 * b + i)];
    };
    if (m == 64) {
        read(0, 0);
        wh_static_for<4>([&](auto bb) {
            constexpr int b = decltype(bb)::value;
            if constexpr (b < 3) read((b + 1) & 1, b + 1);
            __builtin_amdgcn_sched_barrier(0);
            wh_static_for<16>([&](auto ii) { f(bb, ii, x[b & 1][decltype(ii)::value]); });
            __builtin_amdgcn_sched_barrier(0);
        });
    } else {
        wh_static_for<4>([&](auto bb) {
            constexpr int b = decltype(bb)::value;
            if (16 * b < m) {
                read(0, b);  // past the last key: earlier bytes of the tile, not used
                wh_static_for<16>([&](auto ii) {
                    if (16 * b + decltype(ii)::value < m) f(bb, ii, x[0][decltype(ii)::value]);
                });
            }
        });
    }
}

// The inverse RoPE of dim d = 64 blockIdx.x + lane at token_pos
// (E/compute.rs:4160-4197).
struct wh_attn_rope {
    float sn, cs;
    bool any, on;  // the workgroup's dims (uniform) and this one are rope dims
};
__device__ __forceinline__ wh_attn_rope wh_attn_rope_of(const wh_attn_args& a, const wh_attn_pos& v, uint32_t d) {
    wh_attn_rope r{0.0f, 1.0f, false, false};
    const uint32_t first = blockIdx.x * 64, p = (d - a.nope_dim) / 2;
    r.any = first + 63 >= a.nope_dim && first < a.nope_dim + 2 * a.pairs;
    if (r.any) {
        r.on = d >= a.nope_dim && p < a.pairs;
        const float ang = (float)v.token_pos * (r.on ? a.inv_freqs[p] : 0.0f);
        r.sn = -wh_sincosf_glibc(ang, 0);
        r.cs = wh_sincosf_glibc(ang, 1);
    }
    return r;
}

// acc / den when den > 0, then the inverse RoPE; the lanes of a pair
// exchange their values.
__device__ __forceinline__ void wh_attn_finish(const wh_attn_args& a, const wh_attn_pos& v, const wh_attn_rope& rp,
                                               float acc, float den, uint32_t h, uint32_t d) {
    if (den > 0.0f) acc = acc / den;
    if (rp.any) {
        const float other = __shfl_xor(acc, 1, 64);
        if (rp.on) acc = (d & 1) ? other * rp.sn + acc * rp.cs : acc * rp.cs - other * rp.sn;
    }
    if (h < a.heads) v.out[(size_t)h * a.head_dim + d] = acc;
}

// The rest of the window loop for 4 heads x 64 dims per workgroup (grid
// (head_dim / 64, ceil(heads / 4), positions), 256 threads, 4 * wts_ld floats
// of dynamic LDS; wave w = head, lane = dim):
//   max = the largest score (NaN scores never win, E/compute.rs:4125-4127);
//   w_j = expf(score_j - max); denom = expf(sink - max) (if a sink) +
//   (sequential sum of w_j); out_d = sequential sum of w_j * key_j[d] from 0;
//   out_d /= denom when denom > 0; then the inverse RoPE.
// For few positions: each of the head_dim / 64 workgroups of a head makes its
// weights again and, beside its chain of weighted keys, the denominator's,
// which costs less than a launch: four instructions a key.
__global__ void __launch_bounds__(256) k_attn_combine(wh_attn_args a) {
    extern __shared__ __align__(16) float wts[];  // [4][wts_ld]
    __shared__ __align__(16) float tile[2][64 * 64];
    const wh_attn_pos v = wh_attn_resolve(a, blockIdx.z);
    const uint32_t t = threadIdx.x, wave = t >> 6, lane = t & 63;
    const uint32_t h = blockIdx.y * 4 + wave, d = blockIdx.x * 64 + lane;
    const uint32_t nk = v.n_win + v.n_comp;
    const bool hon = h < a.heads;
    const uint32_t hc = hon ? h : a.heads - 1;
    const float sink = a.sink ? a.sink[hc] : 0.0f;
    float* w = wts + wave * a.wts_ld;
    const float* sc = v.scores + (size_t)hc * nk;
    float mx = -__uint_as_float(0x7f800000u);
    // four scores' loads at a time
    for (uint32_t j = lane; j < nk; j += 256) {
        float sv[4];
#pragma unroll
        for (int k = 0; k < 4; ++k) sv[k] = sc[j + 64 * k < nk ? j + 64 * k : j];
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            if (j + 64 * k < nk) w[j + 64 * k] = sv[k];
            mx = fmaxf(mx, sv[k]);
        }
    }
    wh_attn_tiles tiles;
    tiles.start(a, v, nk);
    mx = wh_wave_max(mx);
    for (uint32_t j = lane; j < nk; j += 64) w[j] = wh_expf_glibc(w[j] - mx, kExpTab, kExpfExc, WH_EXPF_EXC_COUNT);
    const float den0 = a.sink ? 0.0f + wh_expf_glibc(sink - mx, kExpTab, kExpfExc, WH_EXPF_EXC_COUNT) : 0.0f;
    float acc = 0.0f, ws = 0.0f;
    tiles.run(a, v, nk, tile, [](auto, uint32_t) {}, [&](auto, const float* tl, uint32_t j0, uint32_t m) {
        float wv[4];  // of 16 keys each
#pragma unroll
        for (int i = 0; i < 4; ++i) wv[i] = w[min(j0 + 16 * i + (lane & 15), nk - 1)];
        const float* tp = tl + lane;
        wh_attn_keys(tp, m, [&](auto bb, auto ii, float x) {
            constexpr int b = decltype(bb)::value, i = decltype(ii)::value;
            ws = ws + wh_mul_bcast<i>(wv[b], 1.0f);
            acc = acc + wh_mul_bcast<i>(wv[b], x);
        });
    });
    wh_attn_finish(a, v, wh_attn_rope_of(a, v, d), acc, den0 + ws, h, d);
}

// The same as two launches, for many positions: the weights once per head ...
// Grid (heads, positions), 256 threads.  The weights replace the scores; the
// denominator waits in the first dim of each 64-dim block of the output,
// which k_attn_weighted's wave of that block reads before it writes.
__global__ void __launch_bounds__(256) k_attn_softmax(wh_attn_args a) {
    constexpr int kPer = WH_ATTN_MAX_KEYS / 256;
    __shared__ __align__(16) wh_osum_lds<WH_ATTN_MAX_KEYS / 32, 32> os;
    __shared__ float red[4];
    const uint32_t t = threadIdx.x, h = blockIdx.x;
    const wh_attn_pos v = wh_attn_resolve(a, blockIdx.y);
    const uint32_t nk = v.n_win + v.n_comp;
    float* sc = v.scores + (size_t)h * nk;
    float x[kPer];
    float mx = -__uint_as_float(0x7f800000u);
#pragma unroll
    for (int k = 0; k < kPer; ++k) x[k] = 256 * k < nk ? sc[min(t + 256 * k, nk - 1)] : mx;
#pragma unroll
    for (int k = 0; k < kPer; ++k) mx = fmaxf(mx, x[k]);
    mx = wh_wave_max(mx);
    if ((t & 63) == 0) red[t >> 6] = mx;
    __syncthreads();
    mx = fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
#pragma unroll
    for (int k = 0; k < kPer; ++k) {
        if (256 * k < nk) {  // uniform
            x[k] = wh_expf_glibc(x[k] - mx, kExpTab, kExpfExc, WH_EXPF_EXC_COUNT);
            if (t + 256 * k < nk) sc[t + 256 * k] = x[k];
        }
    }
    // the weights' sequential sum: one lane up to 512 (as in k_rowpost)
    auto sum = [&](auto l) {
        constexpr int kL = decltype(l)::value;
        auto& s = *(wh_osum_lds<kL, 32>*)&os;
#pragma unroll
        for (int k = 0; k < 32 * kL / 256; ++k) s.rows[wh_osum_at<kL>(t + 256 * k)] = t + 256 * k < nk ? x[k] : -0.0f;
        return wh_ordered_sum_wg<256, kL, 32>(s, 0.0f);
    };
    float ws = 0.0f;
    if (nk <= 512) {
#pragma unroll
        for (int k = 0; k < 2; ++k)
            if (t + 256 * k < nk) os.rows[t + 256 * k] = x[k];
        __syncthreads();
        if (t == 0) ws = wh_ordered_sum_lds(os.rows, nk, 0.0f);
    } else if (nk <= 1024) {
        ws = sum(std::integral_constant<int, 32>());
    } else {
        ws = sum(std::integral_constant<int, WH_ATTN_MAX_KEYS / 32>());
    }
    if (t == 0) {
        const float den0 =
            a.sink ? 0.0f + wh_expf_glibc(a.sink[h] - mx, kExpTab, kExpfExc, WH_EXPF_EXC_COUNT) : 0.0f;
        for (uint32_t b = 0; b < a.head_dim; b += 64) v.out[(size_t)h * a.head_dim + b] = den0 + ws;
    }
}

// ... and the weighted sums: grid (head_dim / 64, ceil(heads / (4 kR)),
// positions), a wave kR heads x 64 dims: two vector instructions per key and
// head, 83% of the launch (64 heads x 628 keys of 32 positions: 63 us and 12 us
// for the weights, 201 us when every 4 heads x 64 dims did both); the wave's
// heads share the key's way through LDS.
template <int kR>
__global__ void __launch_bounds__(256) k_attn_weighted(wh_attn_args a) {
    __shared__ __align__(16) float tile[2][64 * 64];
    const wh_attn_pos v = wh_attn_resolve(a, blockIdx.z);
    const uint32_t t = threadIdx.x, wave = t >> 6, lane = t & 63;
    const uint32_t h0 = (blockIdx.y * 4 + wave) * kR, d = blockIdx.x * 64 + lane;
    const uint32_t nk = v.n_win + v.n_comp;
    wh_attn_tiles tiles;
    tiles.start(a, v, nk);
    const float* w[kR];
    float den[kR], acc[kR];
#pragma unroll
    for (int r = 0; r < kR; ++r) {
        const uint32_t h = h0 + r < a.heads ? h0 + r : a.heads - 1;
        w[r] = v.scores + (size_t)h * nk;
        den[r] = h0 + r < a.heads ? v.out[(size_t)h * a.head_dim + blockIdx.x * 64] : 0.0f;
        acc[r] = 0.0f;
    }
    float wn[2][kR][4];  // the weights of this tile and the next, 16 keys each
    auto weights = [&](float (&d)[kR][4], uint32_t j0) {
#pragma unroll
        for (int r = 0; r < kR; ++r)
#pragma unroll
            for (int i = 0; i < 4; ++i) d[r][i] = w[r][min(j0 + 16 * i + (lane & 15), nk - 1)];
    };
    weights(wn[0], 0);
    tiles.run(
        a, v, nk, tile, [&](auto t0, uint32_t j0) { weights(wn[(decltype(t0)::value + 1) & 1], j0 + 64); },
        [&](auto t0, const float* tl, uint32_t j0, uint32_t m) {
            wh_attn_keys(tl + lane, m, [&](auto bb, auto ii, float x) {
                constexpr int b = decltype(bb)::value, i = decltype(ii)::value;
#pragma unroll
                for (int r = 0; r < kR; ++r)
                    acc[r] = acc[r] + wh_mul_bcast<i>(wn[decltype(t0)::value & 1][r][b], x);
            });
        });
    const wh_attn_rope rp = wh_attn_rope_of(a, v, d);
#pragma unroll
    for (int r = 0; r < kR; ++r) wh_attn_finish(a, v, rp, acc[r], den[r], h0 + r, d);
}
