// A sequential f32 sum by a whole workgroup, bit for bit.
//
// The reference adds long rows of products one after the other in f32
// (hc_pre's dots, the norms' sums of squares), so every rounding depends on
// the one before it, and one lane adds about one term per 8.6 cycles: 59 us
// for 16384 terms.  Here the row is cut into C chunks whose sums run side by
// side from guessed starts, and a result is taken only when every chunk has
// been run from the very value the chunk before it ended with:
//
//   1. guess   an unordered prefix sum gives chunk c's start within a few
//              rounding errors;
//   2. tables  chunk c is added up from eight starts h around the guess, one
//              for each value of the low three mantissa bits: end e(h).
//              Starts that differ by a multiple of 8 ulps go through the same
//              roundings (ties to even included) while the running sum stays
//              near: e(x) = e(h) + (x - h);
//   3. chain   from the true first start, x becomes e(h) + (x - h) chunk by
//              chunk, h the start with x's low bits;
//   4. check   every chunk is added up once more from the x of step 3, all at
//              once.  If each ends, bit for bit, in the next chunk's x, then
//              by induction every x is the sequential sum.  If not, the runs
//              just made replace their entries in the tables, and steps 3 and
//              4 are done again: the chunks up to the first wrong one are
//              right from then on, whatever the values (infinities and NaN
//              too);
//   5. plain   where more than a quarter of the chunks left are wrong, the
//              terms from that group on are added one by one instead.
//
// A round fixes one wrong chunk or more and takes 2.0 us (16384 terms), the
// plain adds of a chunk 0.9 us.  Rows whose neighbouring products cancel to
// 1e-2 or closer would take nearly a round a chunk (their roundings follow the
// terms' grid, not the sum's, so starts 8 ulps apart do not go the same way):
// hc_pre of 4 x 4096 such products 141 us, 68 with step 5, 66 when one lane
// added every row and 22 on N(0, 1) products (2 chunks wrong at first).
//
// On N(0, 1) products 16384 terms take 1.7 rounds on average (the walk meets
// a power of two inside a chunk, where the rounding grid changes), a sum of
// squares 1.0.  Measured launches: hc_pre's 25 sums of 16384 products 58.7 ->
// 15.3 us, the norm of one row of 4096 values 15.3 -> 6.2 us.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

// acc[k] + src[0] + ... + src[kL - 1], one add at a time, for kA sums over
// the same terms; src 16-byte aligned LDS.  Batches of 32 values alternate
// between two register sets, so the next one's reads are in flight.
template <int kL, int kA>
__device__ __forceinline__ void wh_chain_lds(const float* src, float (&acc)[kA]) {
    constexpr int kB = kL < 32 ? kL : 32;  // values per batch
    float4 p[2][kB / 4];
    auto rd = [&](int s, int b) {
#pragma unroll
        for (int i = 0; i < kB / 4; ++i) p[s][i] = *(const float4*)(src + kB * b + 4 * i);
    };
    rd(0, 0);
#pragma unroll
    for (int b = 0; b < kL / kB; ++b) {
        if (b + 1 < kL / kB) rd((b + 1) & 1, b + 1);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int i = 0; i < kB / 4; ++i) {
            const float4 q = p[b & 1][i];
#pragma unroll
            for (int k = 0; k < kA; ++k) acc[k] = acc[k] + q.x;
#pragma unroll
            for (int k = 0; k < kA; ++k) acc[k] = acc[k] + q.y;
#pragma unroll
            for (int k = 0; k < kA; ++k) acc[k] = acc[k] + q.z;
#pragma unroll
            for (int k = 0; k < kA; ++k) acc[k] = acc[k] + q.w;
        }
        __builtin_amdgcn_sched_barrier(0);
    }
}

// The terms of a sum of kC chunks of kL terms in LDS: term i at
// wh_osum_at<kL>(i).  Four floats of padding per chunk keep the lanes' reads,
// one chunk each, in distinct banks.  Terms past the row's end are -0.0f (they
// change no sum).
template <int kL>
__device__ __forceinline__ uint32_t wh_osum_at(uint32_t i) {
    return (i / kL) * (kL + 4) + i % kL;
}
template <int kL, int kC>
struct wh_osum_lds {
    float rows[kC * (kL + 4)];
    float h[kC * 8], e[kC * 8];  // the tables
    float sums[kC];
};

// acc + the terms from chunk c on, one after the other, by one wave: 32 terms
// at a time from two register sets.
template <int kL, int kC>
__device__ __forceinline__ float wh_osum_plain(const wh_osum_lds<kL, kC>& s, int c, float acc) {
    constexpr int kB = kL * kC / 32;
    float4 p[2][8];
    auto rd = [&](int set, int b) {
        const float* src = s.rows + wh_osum_at<kL>(32 * b);
#pragma unroll
        for (int i = 0; i < 8; ++i) p[set][i] = *(const float4*)(src + 4 * i);
    };
    auto add = [&](int set) {
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int i = 0; i < 8; ++i) acc = (((acc + p[set][i].x) + p[set][i].y) + p[set][i].z) + p[set][i].w;
        __builtin_amdgcn_sched_barrier(0);
    };
    int b = c * (kL / 32);
    rd(0, b);
#pragma unroll 1
    for (; b + 1 < kB; b += 2) {
        rd(1, b + 1);
        add(0);
        rd(0, b + 2 < kB ? b + 2 : 0);
        add(1);
    }
    if (b < kB) add(0);
    return acc;
}

// acc0 + term 0 + ... in order, for a workgroup of kT >= 256 threads (all of
// them call; the rows' stores need no barrier before).  kC is 32 or 64.  The
// result is valid in wave 0.
template <int kT, int kL, int kC>
__device__ __forceinline__ float wh_ordered_sum_wg(wh_osum_lds<kL, kC>& s, float acc0) {
    static_assert(kT >= 256 && (kC == 32 || kC == 64) && kL % 32 == 0, "");
    const uint32_t t = threadIdx.x, wave = t >> 6, lane = t & 63;
    // 1. unordered chunk sums: kP threads per chunk
    constexpr int kP0 = kT / kC < 16 ? kT / kC : 16, kP = kP0 < kL / 4 ? kP0 : kL / 4;
    __syncthreads();
    if (t < kC * kP) {
        const float* r = s.rows + (t / kP) * (kL + 4) + (t % kP) * 4;
        float v = 0.0f;
#pragma unroll
        for (int i = 0; i < kL / 4 / kP; ++i) {
            const float4 q = *(const float4*)(r + 4 * kP * i);
            v = v + ((q.x + q.y) + (q.z + q.w));
        }
#pragma unroll
        for (int off = kP / 2; off > 0; off >>= 1) v = v + __shfl_xor(v, off, 64);
        if (t % kP == 0) s.sums[t / kP] = v;
    }
    __syncthreads();
    const uint32_t c = lane % kC;
    const float* row = s.rows + c * (kL + 4);
    if (wave < 4) {
        float incl = s.sums[c];
#pragma unroll
        for (int off = 1; off < kC; off <<= 1) {
            const float o = __shfl_up(incl, off, kC);
            if ((int)c >= off) incl = incl + o;
        }
        const float before = __shfl_up(incl, 1, kC);
        const uint32_t g = __float_as_uint(c ? acc0 + before : acc0) & ~7u;
        // 2. the eight starts over four waves: two sums per lane, or with 32
        // chunks one per half wave
        if constexpr (kC == 64) {
            const float h0 = __uint_as_float(g | (2 * wave)), h1 = __uint_as_float(g | (2 * wave + 1));
            float a[2] = {h0, h1};
            wh_chain_lds<kL, 2>(row, a);
            *(float2*)(s.h + c * 8 + 2 * wave) = make_float2(h0, h1);
            *(float2*)(s.e + c * 8 + 2 * wave) = make_float2(a[0], a[1]);
        } else {
            const uint32_t j = 2 * wave + (lane >> 5);
            float a[1] = {__uint_as_float(g | j)};
            s.h[c * 8 + j] = a[0];
            wh_chain_lds<kL, 1>(row, a);
            s.e[c * 8 + j] = a[0];
        }
    }
    __syncthreads();
    if (wave != 0) return 0.0f;
    // 3. and 4. in wave 0; chunk 8 g + i's start with low bits j is in lane
    // 8 i + j
    int x = 0, from = 0, x_from = __builtin_amdgcn_readfirstlane(__float_as_int(acc0));
    int xc = 0;  // lane c: the start of chunk c
    for (int round = 0; round <= kC; ++round) {
        x = x_from;  // the start of chunk 8 * from, known to be right
        float h = s.h[64 * from + lane], e = s.e[64 * from + lane];
#pragma unroll 1
        for (int g = from; g < kC / 8; ++g) {
            const int nx = ((g + 1) % (kC / 8)) * 64 + lane;
            const float hn = s.h[nx], en = s.e[nx];
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                xc = (int)c == 8 * g + i ? x : xc;
                const float moved = e + (__int_as_float(x) - h);
                const int v = __float_as_int(h) == x ? __float_as_int(e) : __float_as_int(moved);
                x = __builtin_amdgcn_readlane(v, 8 * i + (x & 7));
            }
            h = hn;
            e = en;
        }
        float a[1] = {__int_as_float(xc)};
        wh_chain_lds<kL, 1>(row, a);
        const int next = __shfl_down(xc, 1, 64), end = __float_as_int(a[0]);
        const uint64_t wrong = __ballot(lane < kC && end != (lane == kC - 1 ? x : next));
        if (wrong == 0) break;
        // the chunks up to the first wrong one start right: go on from its group
        from = __builtin_ctzll(wrong) / 8;
        x_from = __builtin_amdgcn_readlane(xc, 8 * from);
        if (4 * __builtin_popcountll(wrong) > kC - 8 * from)
            return wh_osum_plain(s, 8 * from, __int_as_float(x_from));
        if (lane < kC) {
            s.h[c * 8 + (xc & 7)] = __int_as_float(xc);
            s.e[c * 8 + (xc & 7)] = a[0];
        }
        __builtin_amdgcn_wave_barrier();
    }
    return __int_as_float(x);
}
