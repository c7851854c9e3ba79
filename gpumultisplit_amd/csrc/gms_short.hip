// Host engine of the short-input kernels (gms_short.hpp).
#include <algorithm>

#include "gms_short.hpp"

namespace gms {

namespace {

constexpr uint32_t kBlockLds = 160u * 1024u;  // LDS of a CU

uint32_t vec_of(const ShortCall& c) {
    return ((((uintptr_t)c.kin) | ((uintptr_t)c.vin)) & 15u) == 0 ? 1u : 0u;
}

template <int NT, int K, int KW, int VW, class F>
hipError_t block_t(const ShortCall& c, uint32_t bits, const F& f) {
    constexpr size_t lds = 4u * ((size_t)NT * K * (KW + VW) + rank_cnt_words<4, NT>() +
                                 rank_ws_words<4, NT>());
    if constexpr (lds <= kBlockLds) {
        hipLaunchKernelGGL((short_block_kernel<NT, K, KW, VW, F>), dim3(1), dim3(NT), 0, c.stream,
                           c.kin, c.vin, c.kout, c.vout, c.n, bits, f, vec_of(c), c.offs, c.nb);
        return hipGetLastError();
    } else {
        return hipErrorInvalidValue;
    }
}

template <int KW, int VW, class F>
hipError_t block_shape(const ShortCall& c, uint32_t bits, const F& f) {
    if (c.ev) {  // one kernel: all of it counts as the postscan
        for (int i = 0; i < 3; ++i) {
            const hipError_t e = hipEventRecord(c.ev[i], c.stream);
            if (e != hipSuccess) return e;
        }
    }
    // Sorts of 32-bit keys, us: 2000 keys 512 x 4 9.5, 1024 x 4 15.0; 4000 keys 512 x
    // 8 13.0, 1024 x 4 16.4; 5003 keys 512 x 12 16.8, 1024 x 8 20.9; 8000 keys 512 x
    // 16 22.5, 1024 x 8 21.4 (a pass's wave scans cost every wave the same, however
    // few its keys).
    if (c.n <= 1024u) return block_t<256, 4, KW, VW>(c, bits, f);
    if (c.n <= 2048u) return block_t<512, 4, KW, VW>(c, bits, f);
    if (c.n <= 4096u) return block_t<512, 8, KW, VW>(c, bits, f);
    if (c.n <= 6144u) return block_t<512, 12, KW, VW>(c, bits, f);
    return block_t<1024, 8, KW, VW>(c, bits, f);
}

template <int K, int W, int R, int KW, int VW, class F>
hipError_t scatter_t(const ShortCall& c, uint32_t nt, uint32_t* H, uint32_t log_b, uint32_t group,
                     const F& f) {
    hipLaunchKernelGGL((short_scatter_kernel<K, W, R, KW, VW, F>), dim3(nt), dim3(kThreads), 0,
                       c.stream, c.kin, c.vin, c.kout, c.vout, c.n, nt, (const uint32_t*)H, log_b,
                       group, f, vec_of(c), c.offs, c.nb);
    return hipGetLastError();
}

template <int K, int C, int KW, class F>
hipError_t count_t(const ShortCall& c, uint32_t nt, uint32_t* H, uint32_t log_b, const F& f) {
    const dim3 grid((nt + C - 1) / C);
    if constexpr (C == 1) {
        if (log_b <= 3) {
            hipLaunchKernelGGL((short_count_few_kernel<K, KW, F>), grid, dim3(kThreads), 0,
                               c.stream, c.kin, c.n, nt, H, log_b, f, vec_of(c));
            return hipGetLastError();
        }
    }
    if constexpr (KW == 1) {
        if (log_b > 8) {
            hipLaunchKernelGGL((short_count_kernel<K, C, 1024, KW, F>), grid, dim3(kThreads), 0,
                               c.stream, c.kin, c.n, nt, H, log_b, f, vec_of(c));
            return hipGetLastError();
        }
    }
    hipLaunchKernelGGL((short_count_kernel<K, C, 256, KW, F>), grid, dim3(kThreads), 0, c.stream,
                       c.kin, c.n, nt, H, log_b, f, vec_of(c));
    return hipGetLastError();
}

template <int K, int KW, int VW, class F>
hipError_t two_k(const ShortCall& c, const ShortPlan& p, uint32_t* H, const F& f) {
    constexpr uint32_t TILE = kThreads * K;
    const uint32_t nt = (c.n + TILE - 1) / TILE, log_b = p.log_b;
    hipError_t e = c.ev ? hipEventRecord(c.ev[0], c.stream) : hipSuccess;
    if (e != hipSuccess) return e;
    e = p.group == 1 ? count_t<K, 1, KW>(c, nt, H, log_b, f) : count_t<K, 4, KW>(c, nt, H, log_b, f);
    for (int i = 1; i < 3 && c.ev && e == hipSuccess; ++i) e = hipEventRecord(c.ev[i], c.stream);
    if (e != hipSuccess) return e;
    switch (log_b) {
        case 2: return scatter_t<K, 2, 1, KW, VW>(c, nt, H, log_b, p.group, f);
        case 3:
        case 5:
        case 6: return scatter_t<K, 3, 1, KW, VW>(c, nt, H, log_b, p.group, f);
        case 4:
        case 7:
        case 8: return scatter_t<K, 4, 1, KW, VW>(c, nt, H, log_b, p.group, f);
        default: break;
    }
    if constexpr (KW == 1 && VW <= 1) {
        if (log_b == 9) return scatter_t<K, 3, 2, KW, VW>(c, nt, H, log_b, p.group, f);
        if (log_b == 10) return scatter_t<K, 4, 4, KW, VW>(c, nt, H, log_b, p.group, f);
    }
    return hipErrorInvalidValue;
}

template <int KW, int VW, class F>
hipError_t two_shape(const ShortCall& c, const ShortPlan& p, uint32_t* H, const F& f) {
    switch (p.items) {
        case 4: return two_k<4, KW, VW>(c, p, H, f);
        case 8: return two_k<8, KW, VW>(c, p, H, f);
        default: return hipErrorInvalidValue;
    }
}

}  // namespace

// One workgroup while its time stays near that of the two launches it
// replaces (of which the host alone spends 3 us each).  On MI355X, GPU time of
// a key-value call with bucket starts, one workgroup against two launches:
//   8 buckets    1k 3.7 / 5.6 us, 4k 4.8 / 6.1, 8k 6.3 / 6.1
//   256 buckets  1k 4.6 / 6.7 us, 4k 6.6 / 7.4, 8k 9.0 / 7.6
//   1024 buckets 1k 7.8 / 8.1 us, 4k 9.1 / 8.8, 8k 12.4 / 9.2
// so up to 8192 elements, but 4096 where the ids have 9 to 12 bits (a sort's
// 32-bit ids would take four times two launches instead), and 6144 where four
// words per element leave no LDS for more.
bool short_one_block(uint32_t n, uint32_t bits, uint32_t kw, uint32_t vw) {
    return n <= (bits > 8u && bits <= 12u ? 4096u : kw + vw > 3u ? 6144u : 8192u) &&
           form(Form::short_calls, true);
}

// Tiles of 4 elements per thread while that gives at most one tile per CU, then
// 8 (16 keep too few workgroups in flight: below); a count workgroup takes 4
// tiles (C in gms_short.hpp) from the matrix size on where every scatter
// workgroup's reading of all rows costs more than the longer count kernel.  On
// MI355X (GPU us with items.group; key-value, uniform / sorted keys):
//   256 buckets  60k keys 4.1 8.6, 4.4 9.0; 150k 4.1 11.4, 4.4 10.0;
//                600k 8.1 18.6, 8.4 15.2; 1.1M 8.1 27.8 / 28.6, 8.4 17.1 / 19.2, 16.4 18.7 / 25.5
//   64 buckets   300k 8.1 9.8, 8.4 11.4; 1.1M 8.1 15.9 / 17.7, 8.4 13.5 / 15.5, 16.1 16.1 / 22.2;
//                2M 8.1 24.0 / 25.5, 8.4 16.9 / 19.4, 16.4 18.7 / 25.0
//   2 buckets    1.1M 8.1 11.6 / 11.8, 16.1 12.8 / 14.7; 2M 8.1 14.7 / 15.1, 16.1 14.4 / 17.0
static ShortPlan short_shape(uint32_t n, uint32_t log_b) {
    ShortPlan p{n <= (1u << 18) ? 4u : 8u, 1u, log_b, 0u};
    const size_t tile = (size_t)kThreads * p.items;
    const size_t nt = ((size_t)n + tile - 1) / tile;
    if ((nt << log_b) > (p.items == 8u ? 16u * 1024u : 20u * 1024u)) p.group = 4u;
    p.matrix_words = (nt + (p.group > 1u ? (nt + p.group - 1u) / p.group : 0u)) << log_b;
    return p;
}

// The largest short call: where the three stages are as fast.  Key-value,
// uniform / sorted keys, three stages against this: 64 buckets 1.1M 19.0 / 20.8
// and 13.5 / 15.5, 2M 21.0 / 24.8 and 16.9 / 19.4; 2 buckets 2M 15.0 / 15.9 and 14.7 / 15.1;
// 256 buckets 1.3M 22.6 / 25.2 and 18.3 / 19.9, 1.53M 19.5 / 21.4 and 19.6 / 21.0, 2M 23.2 /
// 26.7 and 25.5 / 26.6; 1024 buckets 1M 31.5 and 28.2; 64-bit keys with 32-bit
// values, 256 buckets, 1M 18.9 and 16.9, 1.5M 21.0 and 21.7.
static uint32_t short_top(uint32_t log_b, bool wide) {
    return wide || log_b > 8 ? 1u << 20 : log_b > 6 ? 3u << 19 : 1u << 21;
}

// A whole number of the three stages' tiles has no ragged workgroup, whose
// guarded loads set the time of a call this short: 3 * 2^19 key-value elements
// into 256 buckets take them 16.6 us (1.53M: 19.5) and the two launches 19.4;
// 2 buckets 11.4 and 12.2; 3 * 2^18 into 1024 buckets 21.0 and 24.6.  With 16 to
// 64 buckets the two launches stay ahead (64 buckets 15.3 and 14.2).
static bool whole_tiles_win(uint32_t n, uint32_t log_b) {
    if (n % (uint32_t)(kThreads * tune_items(1, false, false)) != 0) return false;
    return log_b == 10 ? n >= 3u << 18 : (log_b <= 3 || log_b >= 7) && n > 1u << 20;
}

ShortPlan short_plan(uint32_t n, uint32_t num_buckets, uint32_t kw, uint32_t vw) {
    const int cl = ceil_log2_u32(num_buckets);
    const uint32_t lb = cl < 2 ? 2u : (uint32_t)cl;
    const bool wide = kw == 2 || vw == 2;
    if (lb > (wide ? 8u : 10u) || n > short_top(lb, wide) || (!wide && whole_tiles_win(n, lb)) ||
        !form(Form::short_calls, true))
        return ShortPlan{0u, 1u, lb, 0u};
    return short_shape(n, lb);
}

size_t short_matrix_words(uint32_t n_capacity, uint32_t num_buckets) {
    const int cl = ceil_log2_u32(num_buckets);
    const uint32_t lb = cl < 2 ? 2u : (uint32_t)cl;
    if (lb > 10u) return 0;
    // The largest at the ends of the ranges of one tile length.
    size_t m = 0;
    for (uint32_t end : {1u << 18, short_top(lb, false)})
        m = std::max(m, short_shape(n_capacity < end ? n_capacity : end, lb).matrix_words);
    return m;
}

hipError_t launch_short_block(const ShortCall& c, uint32_t bits, const DigitOfF& f) {
    switch (c.vw) {
        case 0: return block_shape<1, 0>(c, bits, f);
        case 1: return block_shape<1, 1>(c, bits, f);
        default: return block_shape<1, 2>(c, bits, f);
    }
}
template <class F>
static hipError_t block64(const ShortCall& c, uint32_t bits, const F& f) {
    switch (c.vw) {
        case 0: return block_shape<2, 0>(c, bits, f);
        case 1: return block_shape<2, 1>(c, bits, f);
        default: return block_shape<2, 2>(c, bits, f);
    }
}
hipError_t launch_short_block(const ShortCall& c, uint32_t bits, const DigitOf64F& f) {
    return block64(c, bits, f);
}
hipError_t launch_short_block(const ShortCall& c, uint32_t bits, const Lite64F& f) {
    return block64(c, bits, f);
}
hipError_t launch_short_sort64(const ShortCall& c) { return block64(c, 64u, RawF64{}); }

hipError_t launch_short_two(const ShortCall& c, const ShortPlan& p, uint32_t* H, const DigitOfF& f) {
    switch (c.vw) {
        case 0: return two_shape<1, 0>(c, p, H, f);
        case 1: return two_shape<1, 1>(c, p, H, f);
        default: return two_shape<1, 2>(c, p, H, f);
    }
}
template <class F>
static hipError_t two64(const ShortCall& c, const ShortPlan& p, uint32_t* H, const F& f) {
    switch (c.vw) {
        case 0: return two_shape<2, 0>(c, p, H, f);
        case 1: return two_shape<2, 1>(c, p, H, f);
        default: return two_shape<2, 2>(c, p, H, f);
    }
}
hipError_t launch_short_two(const ShortCall& c, const ShortPlan& p, uint32_t* H,
                            const DigitOf64F& f) {
    return two64(c, p, H, f);
}
hipError_t launch_short_two(const ShortCall& c, const ShortPlan& p, uint32_t* H, const Lite64F& f) {
    return two64(c, p, H, f);
}

}  // namespace gms

#ifdef GMS_HOST_EMULATION
// Test hook of the CPU emulation build only: the plan of a call, and the matrix
// words of a context for up to n_capacity elements.
extern "C" void gms_emu_short_plan(uint32_t n, uint32_t num_buckets, uint32_t kw, uint32_t vw,
                                   uint32_t* items, uint32_t* group, uint64_t* words) {
    const gms::ShortPlan p = gms::short_plan(n, num_buckets, kw, vw);
    *items = p.items;
    *group = p.group;
    *words = p.matrix_words;
}
extern "C" uint64_t gms_emu_matrix_words(uint32_t n_capacity, uint32_t num_buckets) {
    return gms::matrix_elems(n_capacity, num_buckets);
}
#endif
