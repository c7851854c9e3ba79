// Device-wide histograms of up to 256 bins (the reference's multisplit
// histogram, src/kernels/histogram/multisplit2_histograms.cuh:30-392).
//
// A resident grid (two workgroups per CU) walks full tiles of 256 x 16 words
// with unconditional 16-byte loads, issuing the next tile's loads before it
// counts the current one, so every workgroup keeps a tile in flight while its
// waves add bins into the workgroup's LDS histograms (ds_add).  The ragged ends
// (< one tile) are counted by the last workgroup with guarded loads.  Each workgroup
// folds its sub-histograms and adds its non-zero bins to the global
// histogram once at the end.
#include "gms_internal.hpp"
#include "gms_kernels.hpp"

namespace gms {

constexpr int kHistItems = 16;
constexpr uint32_t kHistTile = kThreads * kHistItems;
constexpr uint32_t kHistGrid = 512;
constexpr uint32_t kRangeGrid = 768;
constexpr int kHistCopies = 32;
constexpr int kRangeCopies = 16;

// bins_of(x, b) maps a register array of words to bins (>= nbins: not
// counted); it sees a whole tile row at once so that a kernel can issue the
// lookups of all its items before it waits for any.  Elements are W words
// (1, or 2 for 64-bit keys): a 16-byte vector of a striped row holds whole
// elements, and bins_of reports an element's bin at its first word and an
// out-of-range bin at its others.  n counts elements.
//
// The workgroup counts into C copies of its histogram, thread t into copy
// t % C, with rows of 257 words so that the copies of one bin lie in different
// banks.  Keys that share a bin across a wave (sorted runs, one dominant bin)
// then add to C addresses instead of one, which the LDS serialises per address;
// evenly spread keys see the same bank spread as with one copy.  Word 256 of a
// row is never read: bins_of may send what is not counted there.
//
// The up to three words before the first 16-byte boundary and the ragged tail
// are counted by the last workgroup, so inputs that start off a boundary (a slice of a
// larger array) take the vector loads too.
template <int W = 1, int C = kHistCopies, bool STREAM = false, class BinsOf>
__device__ __forceinline__ void hist_body(const uint32_t* __restrict__ words, uint32_t num,
                                          uint32_t nbins, uint32_t* __restrict__ d_hist,
                                          BinsOf bins_of) {
    static_assert(W == 1 || W == 2, "elements of 1 or 2 words");
    static_assert(C >= 1 && C <= 64 && (C & (C - 1)) == 0, "copies: a power of two");
    constexpr uint32_t ROW = 257u;
    constexpr uint32_t NH = (uint32_t)C;
    __shared__ uint32_t s_h[NH * ROW];
    const uint32_t tid = threadIdx.x;
    for (uint32_t i = tid; i < NH * ROW; i += kThreads) s_h[i] = 0;
    __syncthreads();
    uint32_t* my = s_h + (tid & (NH - 1u)) * ROW;
    const uint32_t to16 = (uint32_t)((0u - (uint32_t)((uintptr_t)words >> 2)) & 3u) / W;
    const uint32_t head = to16 < num ? to16 : num;
    const uint32_t* p = words + (size_t)head * W;
    const uint32_t n = num - head;
    const uint32_t nfull = (uint32_t)((size_t)n * W / kHistTile);
    uint32_t t = blockIdx.x;
    uint32_t x[kHistItems];
    if (t < nfull) load_striped4_full<kHistItems, true, STREAM>(p, (size_t)t * kHistTile, x);
    // The first tile arrives before the loop: with it possibly pending at the
    // loop's head, the compiler waits there, in every iteration, for the loads
    // that the iteration has just issued, and nothing is prefetched.
    wait_loads();
    while (t < nfull) {
        const uint32_t tn = t + gridDim.x;
        uint32_t y[kHistItems];
        if (tn < nfull) load_striped4_full<kHistItems, true, STREAM>(p, (size_t)tn * kHistTile, y);
        uint32_t b[kHistItems];
        bins_of(x, b);
#pragma unroll
        for (int k = 0; k < kHistItems; ++k)
            if (b[k] <= 256u) atomicAdd(&my[b[k]], 1u);
#pragma unroll
        for (int k = 0; k < kHistItems; ++k) x[k] = y[k];
        t = tn;
    }
    if (blockIdx.x == gridDim.x - 1u) {
        const uint32_t tail = n - nfull * (kHistTile / W), rest = head + tail;
        // Rows of kThreads elements with guarded loads, the row count that of u's array.
        auto ragged = [&](uint32_t i0, auto& u) {
            constexpr int N = (int)(sizeof(u) / sizeof(u[0]));
            uint32_t b[N];
#pragma unroll
            for (int k = 0; k < N; k += W) {
                const uint32_t i = i0 + (uint32_t)(k / W) * kThreads + tid;
                const size_t e = i < head ? i : (size_t)num - tail + (i - head);
#pragma unroll
                for (int w = 0; w < W; ++w) u[k + w] = i < rest ? words[e * W + w] : 0u;
            }
            bins_of(u, b);
#pragma unroll
            for (int k = 0; k < N; ++k)
                if (i0 + (uint32_t)(k / W) * kThreads + tid < rest && b[k] <= 256u)
                    atomicAdd(&my[b[k]], 1u);
        };
        // Few rows do without a tile's 16 guarded loads and lookups, most of them idle: 300
        // samples into 256 edges' bins 4.6 us, 3.4 with four rows.
        if (rest <= 4u * kThreads) {
            uint32_t u[4 * W];
            if (rest) ragged(0u, u);
        } else {  // a second tile for at most three elements
            for (uint32_t i0 = 0; i0 < rest; i0 += kHistTile / W) ragged(i0, x);
        }
    }
    __syncthreads();
    for (uint32_t b = tid; b < nbins; b += kThreads) {
        uint32_t s = 0;
#pragma unroll
        for (uint32_t q = 0; q < NH; ++q) s += s_h[q * ROW + b];
        if (s) atomicAdd(&d_hist[b], s);
    }
}

// Adapts a per-word bin function to hist_body.
template <class F>
__device__ __forceinline__ auto per_word(F f) {
    return [f](auto& x, auto& b) {
        constexpr int N = (int)(sizeof(x) / sizeof(x[0]));
#pragma unroll
        for (int k = 0; k < N; ++k) b[k] = f(x[k]);
    };
}

// STREAM: streamed loads, for inputs of at least kStreamLoadMin words (each
// line is read once and the input is larger than the caches).
template <bool STREAM, class F>
__global__ __launch_bounds__(kThreads) void hist_u32_kernel(const uint32_t* __restrict__ kin,
                                                            uint32_t n, uint32_t nbins,
                                                            uint32_t* __restrict__ d_hist, F f) {
    hist_body<1, kHistCopies, STREAM>(kin, n, nbins, d_hist,
                                           per_word([&](uint32_t k) { return f(k); }));
}

template <bool STREAM>
__global__ __launch_bounds__(kThreads) void hist_even_f32_kernel(const uint32_t* __restrict__ xbits,
                                                                 uint32_t n, uint32_t nbins,
                                                                 uint32_t* __restrict__ d_hist,
                                                                 float lower, float inv_delta) {
    hist_body<1, kHistCopies, STREAM>(xbits, n, nbins, d_hist, per_word([&](uint32_t w) {
        const float d = __uint_as_float(w) - lower;
        // The product is rounded on its own (no contraction with a later add);
        // negative, NaN and >= nbins samples map to an out-of-range bin.
        const float s = __fmul_rn(d, inv_delta);
        return (d >= 0.0f && s < (float)nbins) ? (uint32_t)s : 0xFFFFFFFFu;
    }));
}

// Custom bin edges (the reference's multisplit2_histogram_range_*,
// multisplit2_histograms.cuh:397-699, compared there with CUB's
// HistogramRange): bin i = [levels[i], levels[i+1]); samples outside
// [levels[0], levels[nl-1]) and NaN are not counted.
//
// Every workgroup first builds a table over kRangeCells equal cells of
// [levels[0], levels[nl-1]): cell c holds lo_c = #{interior edges j with
// cell(levels[j]) < c}, cnt_c = #{j : cell(levels[j]) == c} and, for cnt_c = 1,
// that edge.  cell() is non-decreasing and the same function is applied to
// samples and edges, so for a sample x in cell c every edge in a lower cell is
// < x and every edge in a higher one is > x: its bin lies in [lo_c, lo_c + cnt_c].
// Two LDS reads and one compare, bin = lo_c + (x >= edge), settle every sample
// whose cell has at most one edge (an empty cell holds an edge above all
// samples); the others search the cell's edges in LDS.  With 257 random edges
// one wave row in nine has such a sample.  A table of lo_c and cnt_c alone,
// with a search of as many steps as the fullest cell needs for every sample,
// took 72 us for 2^26 and 136 us for 2^27 samples on MI355X (sorted samples 92 and
// 167), this one 62 and 108 (56 and 97).
//
// Building the table takes a workgroup several microseconds.  Inputs of at most
// one tile per workgroup do without it (TABLE = false): a branch-free search of
// eight steps over the edges for every sample.
constexpr uint32_t kRangeCells = 4096;
static_assert(kRangeCells == 16u * kThreads, "16 cells per thread");

template <class T>
struct RangeCellF;

// float: t = (x - lower) * (cells / (upper - lower)), each operation rounded
// on its own and each monotone, truncated and clamped to a cell.
template <>
struct RangeCellF<float> {
    float lower, scale;
    __device__ RangeCellF(float lo, float hi)
        : lower(lo), scale(__fdiv_rn((float)kRangeCells, __fsub_rn(hi, lo))) {}
    __device__ uint32_t operator()(float x) const {
        const float t = __fmul_rn(__fsub_rn(x, lower), scale);
        return t > 0.0f ? (t < (float)kRangeCells ? (uint32_t)t : kRangeCells - 1u) : 0u;
    }
    __device__ static float pad() { return __builtin_inff(); }
};

// uint32: cells of 2^shift keys from lower.
template <>
struct RangeCellF<uint32_t> {
    uint32_t lower, shift;
    __device__ RangeCellF(uint32_t lo, uint32_t hi) : lower(lo), shift(0) {
        const uint32_t r1 = hi - lo - 1u;  // largest x - lower of an in-range x
        const uint32_t bits = r1 ? 32u - (uint32_t)__builtin_clz(r1) : 0u;
        shift = bits > 12u ? bits - 12u : 0u;
    }
    __device__ uint32_t operator()(uint32_t x) const {
        const uint32_t c = (x - lower) >> shift;
        return c < kRangeCells ? c : kRangeCells - 1u;
    }
    __device__ static uint32_t pad() { return 0xFFFFFFFFu; }
};
static_assert(kRangeCells == (1u << 12), "the integer cell shift assumes 2^12 cells");

template <class T>
__device__ __forceinline__ uint32_t bits_of(T v) {
    uint32_t w;
    __builtin_memcpy(&w, &v, sizeof w);
    return w;
}
template <class T>
__device__ __forceinline__ T value_of(uint32_t w) {
    T v;
    __builtin_memcpy(&v, &w, sizeof v);
    return v;
}

template <class T, bool TABLE, bool STREAM>
__global__ __launch_bounds__(kThreads) void hist_range_kernel(const uint32_t* __restrict__ xbits,
                                                              uint32_t n, uint32_t nl,
                                                              const T* __restrict__ d_levels,
                                                              uint32_t* __restrict__ d_hist) {
    constexpr uint32_t CELLS = TABLE ? kRangeCells : 4u;
    __shared__ __attribute__((aligned(16))) uint32_t s_cell[CELLS];  // lo_c | cnt_c << 16
    __shared__ __attribute__((aligned(16))) uint32_t s_edge[CELLS];
    __shared__ T s_lv[256];  // levels[i] for i < nb, then the pad
    __shared__ uint32_t s_ws[kWaves];
    const uint32_t tid = threadIdx.x, nb = nl - 1u;  // nb <= 256: one edge per thread
    const T lo_edge = d_levels[0], hi_edge = d_levels[nb];
    const T pad = RangeCellF<T>::pad();
    const T lv = tid < nb ? d_levels[tid] : pad;
    s_lv[tid] = lv;
    const RangeCellF<T> cell(lo_edge, hi_edge);
    if constexpr (TABLE) {
        // A thread's 16 cells as four 16-byte vectors, in an order that spreads
        // the lanes over the banks.
        uint4* row = reinterpret_cast<uint4*>(s_cell) + 4u * tid;
        const uint32_t pw = bits_of<T>(pad);
#pragma unroll
        for (uint32_t i = 0; i < 4; ++i) {
            const uint32_t r = (i + (tid >> 2)) & 3u;
            row[r] = make_uint4(0u, 0u, 0u, 0u);
            reinterpret_cast<uint4*>(s_edge)[4u * tid + r] = make_uint4(pw, pw, pw, pw);
        }
        __syncthreads();
        const bool interior = tid > 0u && tid < nb;
        const uint32_t mine = interior ? cell(lv) : 0u;
        if (interior) atomicAdd(&s_cell[mine], 1u);
        __syncthreads();
        // Sums of the vectors in cell order, then their exclusive prefixes.
        uint4 v[4];
        uint32_t part[4], sum = 0;
#pragma unroll
        for (uint32_t i = 0; i < 4; ++i) {
            const uint32_t r = (i + (tid >> 2)) & 3u;
            v[i] = row[r];
            const uint32_t q = v[i].x + v[i].y + v[i].z + v[i].w;
#pragma unroll
            for (uint32_t j = 0; j < 4; ++j) part[j] = j == r ? q : part[j];
            sum += q;
        }
        uint32_t total;
        const uint32_t run = block_excl_scan<kWaves>(sum, s_ws, total);
#pragma unroll
        for (uint32_t i = 0; i < 4; ++i) {
            const uint32_t r = (i + (tid >> 2)) & 3u;
            uint32_t a = run;
#pragma unroll
            for (uint32_t j = 0; j < 3; ++j) a += j < r ? part[j] : 0u;
            const uint32_t b = a + v[i].x, c = b + v[i].y, d = c + v[i].z;
            row[r] = make_uint4(a | (v[i].x << 16), b | (v[i].y << 16), c | (v[i].z << 16),
                                d | (v[i].w << 16));
        }
        __syncthreads();
        if (interior && s_cell[mine] >> 16 == 1u) s_edge[mine] = bits_of<T>(lv);
    }
    // (hist_body's first barrier orders the table and the levels before any lookup)
    hist_body<1, kRangeCopies, STREAM>(xbits, n, nb, d_hist, [&](auto& x, auto& b) {
        constexpr int N = (int)(sizeof(x) / sizeof(x[0]));
        if constexpr (TABLE) {
            uint32_t e[N], g[N];
#pragma unroll
            for (int k = 0; k < N; ++k) {
                const uint32_t c = cell(value_of<T>(x[k]));  // any word maps to a cell
                e[k] = s_cell[c];
                g[k] = s_edge[c];
            }
#pragma unroll
            for (int k = 0; k < N; ++k) {
                const T v = value_of<T>(x[k]);
                const uint32_t cnt = e[k] >> 16, lo = e[k] & 0xFFFFu;
                b[k] = lo + (v >= value_of<T>(g[k]) ? 1u : 0u);
                if (cnt > 1u) {  // the number of the cell's edges that are <= v
                    uint32_t l = 0, h = cnt;
                    while (l < h) {
                        const uint32_t m = (l + h) >> 1;
                        if (v >= s_lv[lo + 1u + m]) l = m + 1u;
                        else h = m;
                    }
                    b[k] = lo + l;
                }
            }
        } else {
#pragma unroll
            for (int k = 0; k < N; ++k) b[k] = 0;
#pragma unroll
            for (uint32_t h = 128; h; h >>= 1) {
#pragma unroll
                for (int k = 0; k < N; ++k) b[k] += value_of<T>(x[k]) >= s_lv[b[k] + h] ? h : 0u;
            }
        }
#pragma unroll
        for (int k = 0; k < N; ++k) {
            const T v = value_of<T>(x[k]);
            if (!(v >= lo_edge && v < hi_edge)) b[k] = 256u;  // outside, or NaN: not counted
        }
    });
}

// 64-bit keys through a 64-bit identifier: the same prefetching resident
// grid over the key array viewed as words, each (low, high) word pair one key.
template <bool STREAM>
__global__ __launch_bounds__(kThreads) void hist_u64_kernel(const uint32_t* __restrict__ words,
                                                            uint32_t n, uint32_t nbins,
                                                            uint32_t* __restrict__ d_hist, AnyF64 f) {
    hist_body<2, kHistCopies, STREAM>(words, n, nbins, d_hist, [&](auto& x, auto& b) {
        constexpr int N = (int)(sizeof(x) / sizeof(x[0]));
#pragma unroll
        for (int k = 0; k < N; k += 2) {
            b[k] = f((uint64_t)x[k] | ((uint64_t)x[k + 1] << 32));
            b[k + 1] = 0xFFFFFFFFu;
        }
    });
}

// A workgroup per full tile and one for the ragged ends, if there are any, up to the
// resident grid.
static uint32_t hist_grid(const void* in, uint32_t n, uint32_t max_grid = kHistGrid,
                          uint32_t words = 1) {
    const size_t total = (size_t)n * words, full = total / kHistTile;
    const bool ragged = full * kHistTile != total || ((uintptr_t)in & 15u) != 0;
    const size_t grid = full + (ragged ? 1 : 0);
    return grid < 1 ? 1u : grid < max_grid ? (uint32_t)grid : max_grid;
}

static bool stream_words(size_t words) { return words >= kStreamLoadMin; }

hipError_t launch_histogram_u64(const uint64_t* keys, uint32_t n, uint32_t* d_hist,
                                uint32_t nbins, const AnyF64& f, hipStream_t stream) {
    const uint32_t grid = hist_grid(keys, n, kHistGrid, 2);
    const uint32_t* w = reinterpret_cast<const uint32_t*>(keys);
    if (stream_words((size_t)n * 2))
        hipLaunchKernelGGL((hist_u64_kernel<true>), dim3(grid), dim3(kThreads), 0, stream, w, n,
                           nbins, d_hist, f);
    else
        hipLaunchKernelGGL((hist_u64_kernel<false>), dim3(grid), dim3(kThreads), 0, stream, w, n,
                           nbins, d_hist, f);
    return hipGetLastError();
}

template <class F>
static hipError_t launch_hist(const uint32_t* kin, uint32_t n, uint32_t* d_hist, uint32_t nbins,
                              const F& f, hipStream_t stream) {
    if (stream_words(n))
        hipLaunchKernelGGL((hist_u32_kernel<true, F>), dim3(hist_grid(kin, n)), dim3(kThreads), 0,
                           stream, kin, n, nbins, d_hist, f);
    else
        hipLaunchKernelGGL((hist_u32_kernel<false, F>), dim3(hist_grid(kin, n)), dim3(kThreads), 0,
                           stream, kin, n, nbins, d_hist, f);
    return hipGetLastError();
}

hipError_t launch_histogram_u32(const uint32_t* kin, uint32_t n, uint32_t* d_hist, uint32_t nbins,
                                gms_bucket_desc d, hipStream_t stream) {
    switch (d.kind) {
        case GMS_BUCKET_RANGE: return launch_hist(kin, n, d_hist, nbins, RangeF{nbins}, stream);
        case GMS_BUCKET_DELTA:
            return launch_hist(kin, n, d_hist, nbins, DeltaF::make(d.param, nbins), stream);
        case GMS_BUCKET_DIGIT:
            return launch_hist(kin, n, d_hist, nbins,
                               DigitF{d.param, d.width ? (1u << d.width) - 1u : nbins - 1u}, stream);
        case GMS_BUCKET_LOWBITS:
            return launch_hist(kin, n, d_hist, nbins, DigitF{0u, (1u << d.param) - 1u}, stream);
        case GMS_BUCKET_IDENTITY: return launch_hist(kin, n, d_hist, nbins, IdentF{nbins - 1u}, stream);
        default: return hipErrorInvalidValue;
    }
}

template <class T>
static hipError_t launch_range(const void* x, uint32_t n, int32_t* d_hist, uint32_t num_levels,
                               const T* d_levels, hipStream_t stream) {
    const uint32_t* xb = reinterpret_cast<const uint32_t*>(x);
    uint32_t* h = reinterpret_cast<uint32_t*>(d_hist);
    const dim3 grid(hist_grid(x, n, kRangeGrid)), block(kThreads);
    if (!form(Form::range_table, n / kHistTile >= kRangeGrid))
        hipLaunchKernelGGL((hist_range_kernel<T, false, false>), grid, block, 0, stream, xb, n,
                           num_levels, d_levels, h);
    else if (!stream_words(n))
        hipLaunchKernelGGL((hist_range_kernel<T, true, false>), grid, block, 0, stream, xb, n,
                           num_levels, d_levels, h);
    else
        hipLaunchKernelGGL((hist_range_kernel<T, true, true>), grid, block, 0, stream, xb, n,
                           num_levels, d_levels, h);
    return hipGetLastError();
}

hipError_t launch_histogram_range_f32(const float* x, uint32_t n, int32_t* d_hist,
                                      uint32_t num_levels, const float* d_levels,
                                      hipStream_t stream) {
    return launch_range<float>(x, n, d_hist, num_levels, d_levels, stream);
}

hipError_t launch_histogram_range_u32(const uint32_t* x, uint32_t n, int32_t* d_hist,
                                      uint32_t num_levels, const uint32_t* d_levels,
                                      hipStream_t stream) {
    return launch_range<uint32_t>(x, n, d_hist, num_levels, d_levels, stream);
}

hipError_t launch_histogram_even_f32(const float* x, uint32_t n, int32_t* d_hist, uint32_t nbins,
                                     float lower, float inv_delta, hipStream_t stream) {
    const uint32_t* xb = reinterpret_cast<const uint32_t*>(x);
    uint32_t* h = reinterpret_cast<uint32_t*>(d_hist);
    if (stream_words(n))
        hipLaunchKernelGGL((hist_even_f32_kernel<true>), dim3(hist_grid(x, n)), dim3(kThreads), 0,
                           stream, xb, n, nbins, h, lower, inv_delta);
    else
        hipLaunchKernelGGL((hist_even_f32_kernel<false>), dim3(hist_grid(x, n)), dim3(kThreads), 0,
                           stream, xb, n, nbins, h, lower, inv_delta);
    return hipGetLastError();
}

}  // namespace gms
