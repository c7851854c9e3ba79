// Multisplits and sorts of short inputs (host engine: gms_short.hip).
//
// A short call is bound by its launches (about 3 us of host time each on
// MI355X, and as much again between dependent kernels) and by the latency of
// one workgroup's tile, not by bandwidth, so it takes fewer launches and
// shorter tiles than the prescan -> scan -> postscan path:
//   * one workgroup (short_block_kernel): the whole input in one launch.  The
//     elements stay in LDS through all ranking passes, so a radix sort is one
//     launch too, and a multisplit of up to 2^20 buckets needs no matrix;
//   * two launches (short_count_kernel, short_scatter_kernel): the count
//     matrix is small enough for every workgroup of the second launch to sum
//     what it needs of it, so the scan is not a launch of its own.
// Elements are KW key words and VW value words (1 or 2 / 0, 1 or 2).
#pragma once

#include "gms_internal.hpp"
#include "gms_kernels.hpp"
#include "gms_rank.hpp"

namespace gms {

// 64-bit keys as their own ids (the one-workgroup sort of 64-bit keys).
struct RawF64 {
    GMS_HD uint64_t operator()(uint64_t k) const { return k; }
};

template <int KW>
__device__ __forceinline__ auto short_key(const uint32_t* x, int k) {
    if constexpr (KW == 2) return (uint64_t)x[2 * k] | ((uint64_t)x[2 * k + 1] << 32);
    else return x[k];
}

// Digit of the thread's element k: W bits of the id from `shift`; elements past
// the end take the largest digit, so that they stay behind all others.
template <int W, int K, int KW, class F>
__device__ __forceinline__ auto short_digit(const uint32_t (&kx)[K * KW], uint32_t shift,
                                            uint32_t first, uint32_t n, F f) {
    return [=, &kx](int k) {
        constexpr uint32_t DM = (1u << W) - 1u;
        return first + (uint32_t)k < n ? (uint32_t)(f(short_key<KW>(kx, k)) >> shift) & DM : DM;
    };
}

// Element words in LDS: word w of element i at s[w * TILE + i].
template <int K, int KW, int VW, uint32_t TILE>
__device__ __forceinline__ void short_put(const uint32_t (&kx)[K * KW],
                                          const uint32_t (&vx)[K * (VW ? VW : 1)],
                                          const uint32_t (&pos)[K], uint32_t* s) {
#pragma unroll
    for (int k = 0; k < K; ++k) {
#pragma unroll
        for (int w = 0; w < KW; ++w) s[(uint32_t)w * TILE + pos[k]] = kx[k * KW + w];
#pragma unroll
        for (int w = 0; w < VW; ++w) s[(uint32_t)(KW + w) * TILE + pos[k]] = vx[k * VW + w];
    }
}
template <int K, int KW, int VW, uint32_t TILE>
__device__ __forceinline__ void short_get(uint32_t (&kx)[K * KW], uint32_t (&vx)[K * (VW ? VW : 1)],
                                          const uint32_t* s) {
    static_assert(K % 4 == 0, "16-byte LDS reads");
    const uint32_t off = threadIdx.x * (uint32_t)K;
#pragma unroll
    for (int w = 0; w < KW + VW; ++w) {
#pragma unroll
        for (int i = 0; i < K / 4; ++i) {
            const uint4 v = *reinterpret_cast<const uint4*>(s + (uint32_t)w * TILE + off + 4 * i);
            const uint32_t y[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                if (w < KW) kx[(4 * i + q) * KW + w] = y[q];
                else vx[(4 * i + q) * VW + (w - KW)] = y[q];
            }
        }
    }
}

// Writes element p of LDS to element g of the output.
template <int KW, int VW, uint32_t TILE>
__device__ __forceinline__ void short_write(uint32_t* __restrict__ kout,
                                            uint32_t* __restrict__ vout, uint32_t g, uint32_t p,
                                            const uint32_t* s) {
    if constexpr (KW == 2)
        *reinterpret_cast<uint2*>(kout + 2 * (size_t)g) = make_uint2(s[p], s[TILE + p]);
    else
        kout[g] = s[p];
    if constexpr (VW == 2)
        *reinterpret_cast<uint2*>(vout + 2 * (size_t)g) =
            make_uint2(s[KW * TILE + p], s[(KW + 1) * TILE + p]);
    else if constexpr (VW == 1)
        vout[g] = s[KW * TILE + p];
}

// ---------------------------------------------------------------------------
// The whole input in one workgroup: stable sort by the `bits`-bit id f(key),
// four bits per pass.  offs: starts of the nb buckets, or NULL (binary search
// in the sorted ids, one bucket per thread at a time).
// ---------------------------------------------------------------------------
template <int NT, int K, int KW, int VW, class F>
__global__ __launch_bounds__(NT) void short_block_kernel(
    const uint32_t* __restrict__ kin, const uint32_t* __restrict__ vin,
    uint32_t* __restrict__ kout, uint32_t* __restrict__ vout, uint32_t n, uint32_t bits, F f,
    uint32_t vec, uint32_t* __restrict__ offs, uint32_t nb) {
    constexpr uint32_t TILE = NT * K;
    __shared__ __attribute__((aligned(16))) uint32_t s_item[TILE * (KW + VW)];
    __shared__ uint32_t s_cnt[rank_cnt_words<4, NT>()];
    __shared__ uint32_t s_ws[rank_ws_words<4, NT>()];
    const uint32_t tid = threadIdx.x, first = tid * (uint32_t)K;
    uint32_t kx[K * KW], vx[K * (VW ? VW : 1)];
    load_words<K * KW>(kin, first * KW, n * KW, vec != 0, kx);
    if constexpr (VW) load_words<K * VW>(vin, first * VW, n * VW, vec != 0, vx);
    for (uint32_t shift = 0;;) {
        uint32_t pos[K];
        rank_digits<4, NT, K>(short_digit<4, K, KW>(kx, shift, first, n, f), pos, s_cnt, s_ws, [] {});
        short_put<K, KW, VW, TILE>(kx, vx, pos, s_item);
        __syncthreads();
        shift += 4u;
        if (shift >= bits) break;
        short_get<K, KW, VW, TILE>(kx, vx, s_item);
    }
#pragma unroll
    for (int j = 0; j < K; ++j) {
        const uint32_t p = (uint32_t)j * NT + tid;
        if (p < n) short_write<KW, VW, TILE>(kout, vout, p, p, s_item);
    }
    if (offs) {
        for (uint32_t b = tid; b < nb; b += NT) {
            uint32_t lo = 0, hi = n;
            while (lo < hi) {
                const uint32_t mid = (lo + hi) >> 1;
                uint32_t id;
                if constexpr (KW == 2)
                    id = (uint32_t)f((uint64_t)s_item[mid] | ((uint64_t)s_item[TILE + mid] << 32));
                else
                    id = f(s_item[mid]);
                if (id < b) lo = mid + 1u;
                else hi = mid;
            }
            offs[b] = lo;
        }
    }
}

// ---------------------------------------------------------------------------
// Two launches.  Tiles of kThreads * K elements; the count matrix is
// tile-major, H[t * 2^log_b + b], so that a tile's row is one coalesced read.
// ---------------------------------------------------------------------------
// A workgroup of the count kernel counts C adjacent tiles and also writes the
// sum of their rows (a group row, behind the tile rows) when C > 1.
//
// LDS counters come in kShortCopies copies (lane l adds to copy l mod copies),
// so that keys which share a bucket across a wave do not all add to one LDS
// address; a counter's copies are one 16-byte read.  Combining such keys over
// the wave with ballots, as the prescan does on long inputs, costs a short
// call more than it saves (2^20 zipf keys, 256 buckets: 22.4 against 14.9 us).
constexpr uint32_t kShortCopies = 4;

template <int K, int C, int MAXB, int KW, class F>
__global__ __launch_bounds__(kThreads) void short_count_kernel(const uint32_t* __restrict__ kin,
                                                               uint32_t n, uint32_t num_tiles,
                                                               uint32_t* __restrict__ H,
                                                               uint32_t log_b, F f, uint32_t vec) {
    constexpr uint32_t TILE = kThreads * K;
    __shared__ __attribute__((aligned(16))) uint32_t s_h[C * MAXB * kShortCopies];
    const uint32_t tid = threadIdx.x, B = 1u << log_b;
    const uint32_t ngroups = (num_tiles + C - 1) / C;
    const uint32_t g = xcd_tile(blockIdx.x, ngroups);
    const uint32_t first = g * (uint32_t)C * TILE;  // < n < 2^32
    const uint32_t left = n - first < (uint32_t)C * TILE ? n - first : (uint32_t)C * TILE;
    const uint32_t* p = kin + (size_t)first * KW;
    uint4* cnt4 = reinterpret_cast<uint4*>(s_h);
    for (uint32_t i = tid; i < (uint32_t)C * B; i += kThreads) cnt4[i] = make_uint4(0u, 0u, 0u, 0u);
    __syncthreads();
    const uint32_t copy = tid & (kShortCopies - 1u);
    constexpr int NV = C * K * KW / 4;  // 16-byte vectors per thread
    if (left == (uint32_t)C * TILE && vec) {  // every load in flight before the first use
        uint4 v[NV];
#pragma unroll
        for (int j = 0; j < NV; ++j)
            v[j] = reinterpret_cast<const uint4*>(p)[(uint32_t)j * kThreads + tid];
#pragma unroll
        for (int j = 0; j < NV; ++j) {
            const uint32_t y[4] = {v[j].x, v[j].y, v[j].z, v[j].w};
            const uint32_t c = 4u * ((uint32_t)j * kThreads + tid) / (TILE * KW);
#pragma unroll
            for (int q = 0; q < 4 / KW; ++q)
                atomicAdd(&s_h[(c * B + f(short_key<KW>(y, q))) * kShortCopies + copy], 1u);
        }
    } else {
        // Every element on its own, all loads in flight (at the last element
        // past the end); one ragged workgroup would otherwise set the time of all.
        uint32_t y[C * K][KW];
#pragma unroll
        for (int i = 0; i < C * K; ++i) {
            const uint32_t e = (uint32_t)i * kThreads + tid, at = e < left ? e : left - 1u;
#pragma unroll
            for (int w = 0; w < KW; ++w) y[i][w] = p[(size_t)at * KW + w];
        }
#pragma unroll
        for (int i = 0; i < C * K; ++i) {
            const uint32_t c = (uint32_t)i * kThreads / TILE;
            if ((uint32_t)i * kThreads + tid < left)
                atomicAdd(&s_h[(c * B + f(short_key<KW>(y[i], 0))) * kShortCopies + copy], 1u);
        }
    }
    __syncthreads();
    for (uint32_t b = tid; b < B; b += kThreads) {
        uint32_t sum = 0;
#pragma unroll
        for (int c = 0; c < C; ++c) {
            const uint4 v = cnt4[(uint32_t)c * B + b];
            const uint32_t x = v.x + v.y + v.z + v.w;
            const uint32_t t = g * (uint32_t)C + (uint32_t)c;
            if (t < num_tiles) H[(size_t)t * B + b] = x;
            sum += x;
        }
        if (C > 1) H[(size_t)(num_tiles + g) * B + b] = sum;
    }
}

// The same for at most 8 buckets and one tile per workgroup: byte counters in
// registers, summed over the wave with DPP.  64 lanes on 8 or 16 LDS words
// would serialise (2 buckets, 4M keys: 8.1 us with LDS counters).
template <int K, int KW, class F>
__global__ __launch_bounds__(kThreads) void short_count_few_kernel(
    const uint32_t* __restrict__ kin, uint32_t n, uint32_t num_tiles, uint32_t* __restrict__ H,
    uint32_t log_b, F f, uint32_t vec) {
    constexpr uint32_t TILE = kThreads * K;
    constexpr int NV = K * KW / 4;
    static_assert(K <= 255, "byte counters");
    __shared__ uint32_t s_w[kWaves * 4];
    const uint32_t tid = threadIdx.x, lane = tid & 63u, wid = tid >> 6;
    const uint32_t t = xcd_tile(blockIdx.x, num_tiles);
    const uint32_t nvalid = tile_valid(n, t, TILE);
    const uint32_t* p = kin + (size_t)t * TILE * KW;
    uint64_t c = 0;
    if (nvalid == TILE && vec) {
        uint4 v[NV];
#pragma unroll
        for (int j = 0; j < NV; ++j)
            v[j] = reinterpret_cast<const uint4*>(p)[(uint32_t)j * kThreads + tid];
#pragma unroll
        for (int j = 0; j < NV; ++j) {
            const uint32_t y[4] = {v[j].x, v[j].y, v[j].z, v[j].w};
#pragma unroll
            for (int q = 0; q < 4 / KW; ++q) c += (uint64_t)1 << (8u * f(short_key<KW>(y, q)));
        }
    } else {
        uint32_t y[K][KW];
#pragma unroll
        for (uint32_t i = 0; i < (uint32_t)K; ++i) {
            const uint32_t e = tid + i * kThreads, at = e < nvalid ? e : nvalid - 1u;
#pragma unroll
            for (int w = 0; w < KW; ++w) y[i][w] = p[(size_t)at * KW + w];
        }
#pragma unroll
        for (uint32_t i = 0; i < (uint32_t)K; ++i)
            if (tid + i * kThreads < nvalid) c += (uint64_t)1 << (8u * f(short_key<KW>(y[i], 0)));
    }
    // Buckets j and j + 4 in one word.
    const uint32_t lo = (uint32_t)c, hi = (uint32_t)(c >> 32);
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const uint32_t s = wave_incl_scan(((lo >> (8 * j)) & 255u) | (((hi >> (8 * j)) & 255u) << 16));
        if (lane == 63u) s_w[wid * 4u + (uint32_t)j] = s;
    }
    __syncthreads();
    if (tid < (1u << log_b)) {
        uint32_t s = 0;
#pragma unroll
        for (uint32_t w = 0; w < (uint32_t)kWaves; ++w) s += s_w[w * 4u + (tid & 3u)];
        H[((size_t)t << log_b) + tid] = tid < 4u ? s & 0xFFFFu : s >> 16;
    }
}

// W: bits per ranking pass; R: buckets per thread in the scans (2^log_b <=
// R * kThreads, R a power of two).  offs: starts of the nb buckets, or NULL.
//
// Elements with a 64-bit part (PACKED) do not move through the ranking passes:
// one packed word each does, id << 16 | position in the tile, while the words
// wait in LDS in input order and are fetched through the position by the
// write-out.  Their identifier, about 20 instructions on a 64-bit key, is then
// evaluated once per element.
template <int K, int W, int R, int KW, int VW, class F>
__global__ __launch_bounds__(kThreads) void short_scatter_kernel(
    const uint32_t* __restrict__ kin, const uint32_t* __restrict__ vin,
    uint32_t* __restrict__ kout, uint32_t* __restrict__ vout, uint32_t n, uint32_t num_tiles,
    const uint32_t* __restrict__ H, uint32_t log_b, uint32_t group, F f, uint32_t vec,
    uint32_t* __restrict__ offs, uint32_t nb) {
    constexpr uint32_t TILE = kThreads * K;
    constexpr bool PACKED = KW == 2 || VW == 2;
    static_assert(!PACKED || TILE <= 0x10000u, "16-bit positions");
    __shared__ __attribute__((aligned(16))) uint32_t s_item[TILE * (KW + VW)];
    __shared__ __attribute__((aligned(16))) uint32_t s_pk[PACKED ? TILE : 4];
    __shared__ uint32_t s_cnt[rank_cnt_words<W, kThreads>()];
    __shared__ uint32_t s_ws[rank_ws_words<W, kThreads>()];
    __shared__ __attribute__((aligned(16))) uint32_t s_tot[R * kThreads];  // sums of all tiles
    __shared__ __attribute__((aligned(16))) uint32_t s_pre[R * kThreads];  // sums of the tiles before; then deltas
    __shared__ uint32_t s_b0[kWaves], s_b1[kWaves];
    const uint32_t tid = threadIdx.x, lane = tid & 63u, wid = tid >> 6;
    const uint32_t first = tid * (uint32_t)K;
    const uint32_t t = xcd_tile(blockIdx.x, num_tiles);
    const uint32_t nvalid = tile_valid(n, t, TILE);
    const uint32_t B = 1u << log_b;
    uint32_t kx[K * KW], vx[K * (VW ? VW : 1)];
    load_words<K * KW>(kin + (size_t)t * TILE * KW, first * KW, nvalid * KW, vec != 0, kx);
    if constexpr (VW) load_words<K * VW>(vin + (size_t)t * TILE * VW, first * VW, nvalid * VW, vec != 0, vx);

    // Column sums of the matrix: thread tid adds four adjacent buckets of every
    // G-th row (all rows together are read once per workgroup, 16 bytes per lane).
    uint32_t cnt[R];
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const uint32_t b = tid * (uint32_t)R + (uint32_t)r;
        cnt[r] = b < B ? H[(size_t)t * B + b] : 0u;
        s_tot[tid * (uint32_t)R + (uint32_t)r] = 0;
        s_pre[tid * (uint32_t)R + (uint32_t)r] = 0;
    }
    __syncthreads();
    {
        const uint32_t lq = log_b - 2u;               // log2 of the 16-byte vectors in a row
        const uint32_t G = (uint32_t)kThreads >> lq;  // rows per step
        const uint32_t q = tid & ((1u << lq) - 1u);
        const uint32_t ng = (num_tiles + group - 1u) / group, tg = t / group;
        const uint4* Hv = reinterpret_cast<const uint4*>(H);
        uint4 a = make_uint4(0u, 0u, 0u, 0u), p = a;
        if (group > 1u) {  // the tile's own group: its earlier tiles' rows
            for (uint32_t row = tg * group + (tid >> lq); row < t; row += G) {
                const uint4 v = Hv[((size_t)row << lq) + q];
                p.x += v.x; p.y += v.y; p.z += v.z; p.w += v.w;
            }
            Hv += (size_t)num_tiles << lq;
        }
        constexpr uint32_t U = 8;  // loads in flight
        for (uint32_t r0 = tid >> lq; r0 < ng; r0 += U * G) {
            uint4 v[U];
#pragma unroll
            for (uint32_t u = 0; u < U; ++u) {
                const uint32_t row = r0 + u * G;
                v[u] = row < ng ? Hv[((size_t)row << lq) + q] : make_uint4(0u, 0u, 0u, 0u);
            }
#pragma unroll
            for (uint32_t u = 0; u < U; ++u) {
                const bool before = r0 + u * G < tg;
                a.x += v[u].x; a.y += v[u].y; a.z += v[u].z; a.w += v[u].w;
                p.x += before ? v[u].x : 0u; p.y += before ? v[u].y : 0u;
                p.z += before ? v[u].z : 0u; p.w += before ? v[u].w : 0u;
            }
        }
        const uint32_t av[4] = {a.x, a.y, a.z, a.w}, pv[4] = {p.x, p.y, p.z, p.w};
#pragma unroll
        for (uint32_t i = 0; i < 4; ++i) {
            if (av[i]) atomicAdd(&s_tot[4u * q + i], av[i]);
            if (pv[i]) atomicAdd(&s_pre[4u * q + i], pv[i]);
        }
    }
    __syncthreads();
    // Bucket starts (scan of the totals) and the tile's local starts (scan of
    // its own counts), finished behind the first ranking pass's barrier.
    uint32_t tot[R], pre[R], st = 0, sc = 0;
#pragma unroll
    for (int r = 0; r < R; ++r) {
        tot[r] = s_tot[tid * (uint32_t)R + (uint32_t)r];
        pre[r] = s_pre[tid * (uint32_t)R + (uint32_t)r];
        st += tot[r];
        sc += cnt[r];
    }
    const uint32_t it = wave_incl_scan(st), ic = wave_incl_scan(sc);
    if (lane == 63u) {
        s_b0[wid] = it;
        s_b1[wid] = ic;
    }
    auto deltas = [&] {
        uint32_t g = it - st, l = ic - sc;
#pragma unroll
        for (uint32_t i = 0; i < (uint32_t)kWaves; ++i) {
            g += i < wid ? s_b0[i] : 0u;
            l += i < wid ? s_b1[i] : 0u;
        }
#pragma unroll
        for (int r = 0; r < R; ++r) {
            const uint32_t b = tid * (uint32_t)R + (uint32_t)r;
            if (offs && t == 0 && b < nb) offs[b] = g;
            s_pre[b] = g + pre[r] - l;  // only this thread read word b
            g += tot[r];
            l += cnt[r];
        }
    };
    if constexpr (PACKED) {
        constexpr uint32_t DM = (1u << W) - 1u;
        uint32_t pk[K], none[1 * K], at[K];
#pragma unroll
        for (int k = 0; k < K; ++k) {
            const uint32_t e = first + (uint32_t)k;
            at[k] = e;
            none[k] = 0;
            // past the end: an id of all ones, behind every other
            pk[k] = (e < nvalid ? f(short_key<KW>(kx, k)) : 0xFFFFu) << 16 | e;
        }
        short_put<K, KW, VW, TILE>(kx, vx, at, s_item);
        for (uint32_t shift = 0;;) {
            uint32_t pos[K];
            rank_digits<W, kThreads, K>([&](int k) { return (pk[k] >> (16u + shift)) & DM; }, pos,
                                        s_cnt, s_ws, [&] { if (shift == 0) deltas(); });
            short_put<K, 1, 0, TILE>(pk, none, pos, s_pk);
            __syncthreads();
            shift += (uint32_t)W;
            if (shift >= log_b) break;
            short_get<K, 1, 0, TILE>(pk, none, s_pk);
        }
#pragma unroll 4
        for (int j = 0; j < K; ++j) {
            const uint32_t p = (uint32_t)j * kThreads + tid;
            if (p < nvalid) {
                const uint32_t w = s_pk[p];
                uint32_t g = s_pre[w >> 16] + p;
                g = g < n ? g : n - 1u;
                short_write<KW, VW, TILE>(kout, vout, g, w & 0xFFFFu, s_item);
            }
        }
        return;
    }
    for (uint32_t shift = 0;;) {
        uint32_t pos[K];
        rank_digits<W, kThreads, K>(short_digit<W, K, KW>(kx, shift, first, nvalid, f), pos, s_cnt,
                                    s_ws, [&] { if (shift == 0) deltas(); });
        short_put<K, KW, VW, TILE>(kx, vx, pos, s_item);
        __syncthreads();
        shift += (uint32_t)W;
        if (shift >= log_b) break;
        short_get<K, KW, VW, TILE>(kx, vx, s_item);
    }
#pragma unroll 4
    for (int j = 0; j < K; ++j) {
        const uint32_t p = (uint32_t)j * kThreads + tid;
        if (p < nvalid) {
            uint32_t id;
            if constexpr (KW == 2)
                id = f((uint64_t)s_item[p] | ((uint64_t)s_item[TILE + p] << 32));
            else
                id = f(s_item[p]);
            uint32_t g = s_pre[id] + p;
            g = g < n ? g : n - 1u;
            short_write<KW, VW, TILE>(kout, vout, g, p, s_item);
        }
    }
}

}  // namespace gms
