// Stable in-workgroup ranking of W-bit digits with the counters in registers.
//
// Thread t of NT holds K consecutive elements of the workgroup's order
// (positions [t*K, t*K+K)) and their digits.  rank_digits gives every element
// its position in the order stably sorted by digit:
//   1. each thread counts its digits in packed registers, which also yields an
//      element's rank among the thread's own elements of its digit;
//   2. the counts, two digits to a 32-bit word, are prefix-summed over the
//      wave with DPP and over the waves through one LDS exchange;
//   3. the thread's starting positions go to its own column of s_cnt, where a
//      dynamic index can reach them: position = column[digit] + rank.
// One barrier.  Only LDS column words of the thread itself are read back, so
// none is needed around step 3.
//
// An LDS counter per (digit, thread) with one ds_add_rtn per key, the form it
// replaces, spends about 13 clocks of the CU's LDS pipe per wave and key on
// MI355X and needs three more barriers; here a key costs vector ALU work, which
// has room to spare.
#pragma once

#include "gms_device.hpp"

namespace gms {

// Packed positions are 16-bit: at most 2^16 elements per workgroup.
template <int W>
constexpr int rank_words() { return W <= 1 ? 1 : 1 << (W - 1); }
// LDS words of the per-thread columns / of the wave exchange.
template <int W, int NT>
constexpr uint32_t rank_cnt_words() { return (uint32_t)rank_words<W>() * NT; }
template <int W, int NT>
constexpr uint32_t rank_ws_words() {
    return (uint32_t)(rank_words<W>() * (NT / 64) < 64 ? 64 : rank_words<W>() * (NT / 64));
}

// Step 1: slot[k] = digit of element k << 8 | its rank among the thread's
// earlier elements of that digit (one register per element until its position
// is known); c[j] = count of digit j (low half) and of digit j + DP (high half).
template <int W, int K, class Digit>
__device__ __forceinline__ void rank_count(Digit digit, uint32_t (&slot)[K],
                                           uint32_t (&c)[rank_words<W>()]) {
    constexpr int DP = rank_words<W>();
    static_assert(W >= 1 && W <= 4, "1 to 4 bits per pass");
    static_assert(K <= 255, "byte counters");
    if constexpr (W <= 2) {  // four byte counters
        uint32_t p = 0;
#pragma unroll
        for (int k = 0; k < K; ++k) {
            const uint32_t d = digit(k), sh = d * 8u;
            slot[k] = ((p >> sh) & 255u) | (d << 8);
            p += 1u << sh;
        }
#pragma unroll
        for (int j = 0; j < DP; ++j)
            c[j] = ((p >> (8 * j)) & 255u) | (((p >> (8 * (j + DP))) & 255u) << 16);
    } else if constexpr (W == 3) {  // eight byte counters
        uint64_t p = 0;
#pragma unroll
        for (int k = 0; k < K; ++k) {
            const uint32_t d = digit(k), sh = d * 8u;
            slot[k] = ((uint32_t)(p >> sh) & 255u) | (d << 8);
            p += (uint64_t)1 << sh;
        }
        const uint32_t lo = (uint32_t)p, hi = (uint32_t)(p >> 32);
#pragma unroll
        for (int j = 0; j < DP; ++j)
            c[j] = ((lo >> (8 * j)) & 255u) | (((hi >> (8 * j)) & 255u) << 16);
    } else {
        // Sixteen 4-bit counters, for groups of at most 15 elements; an
        // element's rank adds the counts of the groups before its own.
        constexpr int NG = (K + 14) / 15, G = (K + NG - 1) / NG;
        uint64_t p[NG];
#pragma unroll
        for (int g = 0; g < NG; ++g) {
            p[g] = 0;
#pragma unroll
            for (int k = g * G; k < (g + 1) * G && k < K; ++k) {
                const uint32_t d = digit(k), sh = d * 4u;
                uint32_t r = d << 8;
#pragma unroll
                for (int q = 0; q <= g; ++q) r += (uint32_t)(p[q] >> sh) & 15u;
                slot[k] = r;
                p[g] += (uint64_t)1 << sh;
            }
        }
#pragma unroll
        for (int j = 0; j < DP; ++j) {
            c[j] = 0;
#pragma unroll
            for (int g = 0; g < NG; ++g)
                c[j] += (((uint32_t)p[g] >> (4 * j)) & 15u) |
                        ((((uint32_t)(p[g] >> 32) >> (4 * j)) & 15u) << 16);
        }
    }
}

// pos[k] for every element; digit(k) gives its digit.  `mid` runs after the barrier (work of the caller
// that needs one).  s_cnt: rank_cnt_words words, s_ws: rank_ws_words words;
// the caller puts a barrier between the use of pos (its scatter) and the next
// call.
template <int W, int NT, int K, class Digit, class Mid>
__device__ __forceinline__ void rank_digits(Digit digit, uint32_t (&pos)[K], uint32_t* s_cnt,
                                            uint32_t* s_ws, Mid mid) {
    constexpr int DP = rank_words<W>();
    constexpr int NW = NT / 64;
    static_assert((uint64_t)NT * K <= 65535u, "16-bit positions");
    const uint32_t tid = threadIdx.x, lane = tid & 63u;
    const uint32_t wid = (uint32_t)GMS_READFIRSTLANE((int)(tid >> 6));
    uint32_t c[DP], inc[DP];
    rank_count<W, K>(digit, pos, c);
#pragma unroll
    for (int j = 0; j < DP; ++j) inc[j] = wave_incl_scan(c[j]);
    if (lane == 63u) {
#pragma unroll
        for (int j = 0; j < DP; ++j) s_ws[j * NW + wid] = inc[j];
    }
    __syncthreads();
    // Every wave scans the (digit pair, wave) totals, PER of them per lane; the
    // high halves start where the low halves end.
    constexpr int PER = (DP * NW + 63) / 64;
    uint32_t w[PER], s = 0;
#pragma unroll
    for (int i = 0; i < PER; ++i) {
        const uint32_t x = lane * (uint32_t)PER + (uint32_t)i;
        w[i] = x < (uint32_t)(DP * NW) ? s_ws[x] : 0u;
        s += w[i];
    }
    const uint32_t si = wave_incl_scan(s);
    uint32_t ex = si - s + (wave_last(si) << 16);
    uint32_t e[PER];
#pragma unroll
    for (int i = 0; i < PER; ++i) {
        e[i] = ex;
        ex += w[i];
    }
    uint32_t* col = s_cnt + tid;
#pragma unroll
    for (int j = 0; j < DP; ++j) {
        const uint32_t x = (uint32_t)(j * NW) + wid;
        uint32_t base = 0;
        if constexpr (PER == 1) {
            base = (uint32_t)GMS_READLANE((int)e[0], (int)x);
        } else {
#pragma unroll
            for (int i = 0; i < PER; ++i) {
                const uint32_t v = (uint32_t)GMS_READLANE((int)e[i], (int)(x / PER));
                base = x % PER == (uint32_t)i ? v : base;
            }
        }
        col[j * NT] = base + inc[j] - c[j];
    }
    mid();
#pragma unroll
    for (int k = 0; k < K; ++k) {
        const uint32_t d = pos[k] >> 8;
        const uint32_t v = col[(d & (uint32_t)(DP - 1)) * (uint32_t)NT];
        pos[k] = (pos[k] & 255u) + ((d & (uint32_t)DP) ? v >> 16 : v & 0xFFFFu);
    }
}

// Bits of the ranking passes of a LOG_B-bit id: one pass up to 4 bits, then
// 3 + 3 (2), 4 + 4 (3), and 3 or 4 bits in three passes.
constexpr int rank_pass_bits(int log_b) { return log_b <= 4 ? log_b : (log_b <= 6 || log_b == 9 ? 3 : 4); }

template <int SHIFT, int W, int NT, int K, bool KV, bool FULL, class F, class Mid>
__device__ __forceinline__ void rank_tile_pass(const uint32_t (&key)[K], const uint32_t (&val)[K],
                                               uint32_t nvalid, F f, uint32_t* s_keys,
                                               uint32_t* s_vals, uint32_t* s_cnt, uint32_t* s_ws,
                                               Mid mid) {
    constexpr uint32_t DM = (1u << W) - 1u;
    const uint32_t first = threadIdx.x * (uint32_t)K;
    uint32_t pos[K];
    rank_digits<W, NT, K>(
        [&](int k) { return FULL || first + (uint32_t)k < nvalid ? (f(key[k]) >> SHIFT) & DM : DM; },
        pos, s_cnt, s_ws, mid);
#pragma unroll
    for (int k = 0; k < K; ++k) {
        s_keys[pos[k]] = key[k];
        if constexpr (KV) s_vals[pos[k]] = val[k];
    }
    __syncthreads();
}

// Leaves the tile's nvalid keys (and values) in s_keys (s_vals), stably sorted
// by the LOG_B-bit id f(key); key and val hold the thread's K consecutive keys
// of the tile.  Keys past nvalid take the largest digit of every pass and stay
// behind.  `mid` runs after the first pass's barrier; ends with a barrier.
template <int LOG_B, int NT, int K, bool KV, bool FULL, class F, class Mid>
__device__ __forceinline__ void rank_tile(uint32_t (&key)[K], uint32_t (&val)[K], uint32_t nvalid,
                                          F f, uint32_t* s_keys, uint32_t* s_vals,
                                          uint32_t* s_cnt, uint32_t* s_ws, Mid mid) {
    constexpr int W = rank_pass_bits(LOG_B);
    rank_tile_pass<0, W, NT, K, KV, FULL>(key, val, nvalid, f, s_keys, s_vals, s_cnt, s_ws, mid);
    auto reload = [&] {
        static_assert(K % 4 == 0, "16-byte LDS reads of whole rows");
        const uint32_t off = threadIdx.x * (uint32_t)K;
#pragma unroll
        for (int i = 0; i < K / 4; ++i) {
            const uint4 a = *reinterpret_cast<const uint4*>(s_keys + off + 4 * i);
            key[4 * i + 0] = a.x; key[4 * i + 1] = a.y; key[4 * i + 2] = a.z; key[4 * i + 3] = a.w;
            if constexpr (KV) {
                const uint4 b = *reinterpret_cast<const uint4*>(s_vals + off + 4 * i);
                val[4 * i + 0] = b.x; val[4 * i + 1] = b.y; val[4 * i + 2] = b.z; val[4 * i + 3] = b.w;
            }
        }
    };
    auto none = [] {};
    if constexpr (LOG_B > W) {
        constexpr int W1 = LOG_B - W < W ? LOG_B - W : W;
        reload();
        rank_tile_pass<W, W1, NT, K, KV, FULL>(key, val, nvalid, f, s_keys, s_vals, s_cnt, s_ws, none);
    }
    if constexpr (LOG_B > 2 * W) {
        constexpr int W2 = LOG_B - 2 * W;
        static_assert(W2 <= W, "at most three passes");
        reload();
        rank_tile_pass<2 * W, W2, NT, K, KV, FULL>(key, val, nvalid, f, s_keys, s_vals, s_cnt, s_ws, none);
    }
}

}  // namespace gms
