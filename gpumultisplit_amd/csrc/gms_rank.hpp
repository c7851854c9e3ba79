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

// Step 1: slot[k] = rank of element k among the thread's earlier elements of
// its digit; c[j] = count of digit j (low half) and of digit j + DP (high half).
template <int W, int K>
__device__ __forceinline__ void rank_count(const uint32_t (&dig)[K], uint32_t (&slot)[K],
                                           uint32_t (&c)[rank_words<W>()]) {
    constexpr int DP = rank_words<W>();
    static_assert(W >= 1 && W <= 4, "1 to 4 bits per pass");
    static_assert(K <= 255, "byte counters");
    if constexpr (W <= 2) {  // four byte counters
        uint32_t p = 0;
#pragma unroll
        for (int k = 0; k < K; ++k) {
            const uint32_t sh = dig[k] * 8u;
            slot[k] = (p >> sh) & 255u;
            p += 1u << sh;
        }
#pragma unroll
        for (int j = 0; j < DP; ++j)
            c[j] = ((p >> (8 * j)) & 255u) | (((p >> (8 * (j + DP))) & 255u) << 16);
    } else if constexpr (W == 3) {  // eight byte counters
        uint64_t p = 0;
#pragma unroll
        for (int k = 0; k < K; ++k) {
            const uint32_t sh = dig[k] * 8u;
            slot[k] = (uint32_t)(p >> sh) & 255u;
            p += (uint64_t)1 << sh;
        }
        const uint32_t lo = (uint32_t)p, hi = (uint32_t)(p >> 32);
#pragma unroll
        for (int j = 0; j < DP; ++j)
            c[j] = ((lo >> (8 * j)) & 255u) | (((hi >> (8 * j)) & 255u) << 16);
    } else if constexpr (K <= 30) {  // sixteen 4-bit counters, for at most 15 elements at a time
        constexpr int G = K <= 15 ? K : (K + 1) / 2;
        uint64_t a = 0, b = 0;
#pragma unroll
        for (int k = 0; k < G; ++k) {
            const uint32_t sh = dig[k] * 4u;
            slot[k] = (uint32_t)(a >> sh) & 15u;
            a += (uint64_t)1 << sh;
        }
#pragma unroll
        for (int k = G; k < K; ++k) {
            const uint32_t sh = dig[k] * 4u;
            slot[k] = ((uint32_t)(a >> sh) & 15u) + ((uint32_t)(b >> sh) & 15u);
            b += (uint64_t)1 << sh;
        }
        const uint32_t al = (uint32_t)a, ah = (uint32_t)(a >> 32);
        const uint32_t bl = (uint32_t)b, bh = (uint32_t)(b >> 32);
#pragma unroll
        for (int j = 0; j < DP; ++j) {
            c[j] = ((al >> (4 * j)) & 15u) | (((ah >> (4 * j)) & 15u) << 16);
            if constexpr (K > G) c[j] += ((bl >> (4 * j)) & 15u) | (((bh >> (4 * j)) & 15u) << 16);
        }
    } else {  // sixteen byte counters in two registers pairs
        uint64_t lo = 0, hi = 0;
#pragma unroll
        for (int k = 0; k < K; ++k) {
            const uint32_t sh = (dig[k] & 7u) * 8u;
            const bool up = (dig[k] & 8u) != 0;
            const uint64_t p = up ? hi : lo;
            slot[k] = (uint32_t)(p >> sh) & 255u;
            const uint64_t q = p + ((uint64_t)1 << sh);
            hi = up ? q : hi;
            lo = up ? lo : q;
        }
#pragma unroll
        for (int j = 0; j < DP; ++j)
            c[j] = ((uint32_t)(lo >> (8 * j)) & 255u) | (((uint32_t)(hi >> (8 * j)) & 255u) << 16);
    }
}

// pos[k] for every element.  `mid` runs after the barrier (work of the caller
// that needs one).  s_cnt: rank_cnt_words words, s_ws: rank_ws_words words;
// the caller puts a barrier between the use of pos (its scatter) and the next
// call.
template <int W, int NT, int K, class Mid>
__device__ __forceinline__ void rank_digits(const uint32_t (&dig)[K], uint32_t (&pos)[K],
                                            uint32_t* s_cnt, uint32_t* s_ws, Mid mid) {
    constexpr int DP = rank_words<W>();
    constexpr int NW = NT / 64;
    static_assert((uint64_t)NT * K <= 65535u, "16-bit positions");
    const uint32_t tid = threadIdx.x, lane = tid & 63u;
    const uint32_t wid = (uint32_t)GMS_READFIRSTLANE((int)(tid >> 6));
    uint32_t c[DP], inc[DP];
    rank_count<W, K>(dig, pos, c);
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
        const uint32_t v = col[(dig[k] & (uint32_t)(DP - 1)) * (uint32_t)NT];
        pos[k] += (dig[k] & (uint32_t)DP) ? v >> 16 : v & 0xFFFFu;
    }
}

}  // namespace gms
