// Multisplit and radix sort of elements with 64-bit keys and/or 64-bit values.
//
// The reference's API is templated on KeyT and ValueT (src/api/multisplit.cuh:
// 81-82, :199-200; src/api/multisplit_sort.cuh:366-527;
// multisplit_sort_pairs.cuh:67-228) although its kernels move 32-bit words.
// Here an element is KW key words and VW value words (KW, VW in {1, 2}, 0 <=
// VW), stored as the caller's arrays of 32- or 64-bit integers.
//
// Same three stages as the 32-bit path (prescan, device scan, postscan) on the
// same histogram matrix layout.  The postscan does not move the element
// through its LDS ranking passes: it ranks one packed word per element,
// bucket << 16 | position in the tile, with the 32-bit ranking code
// (postscan_rank), while the element's words wait in LDS in input order in
// the area the ranking counters used.  The write-out reads the packed word of
// each slot and fetches the element's words through its position, so a
// 16-byte element costs the ranking no more LDS traffic than a 4-byte key.
#include <algorithm>

#include "gms_wide_kernels.hpp"

namespace gms {

uint32_t wide_tile_elems(uint32_t key_words, uint32_t value_words) {
    return kThreads * (uint32_t)wide_items((int)key_words, (int)value_words);
}

uint32_t wide_min_tile_elems() {
    uint32_t m = wide_tile_elems(2, 0);
    for (uint32_t kw = 1; kw <= 2; ++kw)
        for (uint32_t vw = 1; vw <= 2; ++vw)
            if (kw == 2 || vw == 2) m = std::min(m, wide_tile_elems(kw, vw));
    return m;
}

// Calls fn with the identifier of 64-bit keys for one digit (id >> shift) &
// mask of the descriptor's bucket id (shift 0, mask ~0: the id itself).
template <class Fn>
static auto with_id64(const gms_bucket_desc64& d, uint32_t B, uint32_t shift, uint32_t mask, Fn&& fn) {
    if (Lite64F::covers(d.kind)) return fn(Lite64F::make(d.kind, d.param, d.width, B, shift, mask));
    return fn(DigitOf64F{AnyF64::make(d.kind, d.param, d.width, B), shift, mask});
}
// The same for 32-bit keys.
static DigitOfF id32(const gms_bucket_desc64& d, uint32_t B, uint32_t shift, uint32_t mask) {
    return DigitOfF{AnyF::make(d.kind, (uint32_t)d.param, d.width, B), shift, mask};
}

// One pass into B buckets by the digit (id >> shift) & mask of the ids of
// descriptor d for `ids` buckets.
static gms_status wide_stages(Scratch& s, const uint32_t* kin, const uint32_t* vin,
                              uint32_t* kout, uint32_t* vout, uint32_t n, uint32_t kw,
                              uint32_t vw, uint32_t B, const gms_bucket_desc64& d, uint32_t ids,
                              uint32_t shift, uint32_t mask, uint32_t* d_offsets,
                              hipStream_t stream) {
    if (n == 0) return d_offsets ? hip_status(launch_fill(d_offsets, 0u, B, stream)) : GMS_SUCCESS;
    if (B == 1) {
        hipError_t e = launch_copy(kin, kout, (size_t)n * kw, stream);
        if (e == hipSuccess && vw) e = launch_copy(vin, vout, (size_t)n * vw, stream);
        if (e == hipSuccess && d_offsets) e = launch_fill(d_offsets, 0u, 1u, stream);
        return hip_status(e);
    }
    const int lb = ceil_log2_u32(B);
    // Short inputs: one or two launches.
    const bool apart = starts_apart(d_offsets, B, kin, vin, kout, vout, n, kw, vw);
    const bool block = short_one_block(n, (uint32_t)lb, kw, vw);
    const ShortPlan sp = short_plan(n, B, kw, vw);
    if (apart && (block || (sp.items && sp.matrix_words <= s.hist_cap))) {
        const ShortCall c{kin, vin, kout, vout, n, kw, vw, d_offsets, B, stream};
        auto go = [&](const auto& f) {
            return block ? launch_short_block(c, (uint32_t)lb, f) : launch_short_two(c, sp, s.hist, f);
        };
        return hip_status(kw == 2 ? with_id64(d, ids, shift, mask, go) : go(id32(d, ids, shift, mask)));
    }
    const uint32_t tile = wide_tile_elems(kw, vw);
    const uint32_t nt = (uint32_t)(((size_t)n + tile - 1) / tile);
    const size_t m = ((size_t)1 << lb) * nt;
    // One-launch scan when the scratch has its status words (the prescan
    // clears them), else the two-launch one.
    const bool one = s.status && scan_chunks(m) <= s.status_cap;
    if (m > s.hist_cap || (!one && scan_partials_needed(m) > s.part_cap)) return GMS_ERR_CAPACITY;
    auto al16 = [](const void* p) { return p == nullptr || (((uintptr_t)p) & 15u) == 0; };
    WideCall c{kin, vin, kout, vout, n, nt, s.hist, al16(kin) && al16(vin), stream};
    c.offs = apart ? d_offsets : nullptr;
    c.nb = B;
    if (one) {
        c.scan_status = s.status;
        c.scan_chunks = scan_chunks(m);
    }
    auto stage = [&](bool prescan) {
        if (kw == 2) {
            const AnyF64 f = AnyF64::make(d.kind, d.param, d.width, ids);
            return mask == ~0u ? wide_dispatch64(c, lb, vw, f, prescan)
                               : wide_dispatch64(c, lb, vw, DigitOf64F{f, shift, mask}, prescan);
        }
        if (vw != 2) return hipErrorInvalidValue;
        return wide_stage<1, 2>(c, lb, id32(d, ids, shift, mask), prescan);
    };
    hipError_t e = stage(true);
    if (e == hipSuccess)
        e = one ? launch_scan_single(s.hist, s.hist, (uint32_t)m, s.status, stream)
                : launch_exclusive_scan(s.hist, s.hist, (uint32_t)m, s.part, stream);
    if (e == hipSuccess) e = stage(false);
    if (e == hipSuccess && d_offsets && !c.offs)
        e = launch_gather_offsets(s.hist, nt, B, d_offsets, stream);
    return hip_status(e);
}

gms_status run_wide_multisplit(Scratch& s, const uint32_t* kin, const uint32_t* vin,
                               uint32_t* kout, uint32_t* vout, uint32_t n, uint32_t kw,
                               uint32_t vw, uint32_t B, const gms_bucket_desc64& d,
                               uint32_t* d_offsets, hipStream_t stream) {
    return wide_stages(s, kin, vin, kout, vout, n, kw, vw, B, d, B, 0u, ~0u, d_offsets, stream);
}

// Bucket starts read off a finished output.
static gms_status wide_starts(const uint32_t* kout, uint32_t n, uint32_t kw, uint32_t B,
                              const gms_bucket_desc64& d, uint32_t* d_offsets, hipStream_t stream) {
    if (kw == 2)
        return hip_status(launch_bucket_starts<2>(kout, n, B, AnyF64::make(d.kind, d.param, d.width, B),
                                                  d_offsets, stream));
    return hip_status(launch_bucket_starts<1>(kout, n, B,
                                              AnyF::make(d.kind, (uint32_t)d.param, d.width, B),
                                              d_offsets, stream));
}

gms_status run_wide_large(Scratch& s, uint32_t* ktmp, uint32_t* vtmp, const uint32_t* kin,
                          const uint32_t* vin, uint32_t* kout, uint32_t* vout, uint32_t n,
                          uint32_t kw, uint32_t vw, uint32_t B, const gms_bucket_desc64& d,
                          uint32_t* d_offsets, hipStream_t stream) {
    if (n == 0) return d_offsets ? hip_status(launch_fill(d_offsets, 0u, B, stream)) : GMS_SUCCESS;
    const int bits = ceil_log2_u32(B);
    if (short_one_block(n, (uint32_t)bits, kw, vw)) {
        uint32_t* offs = B <= kShortBlockOffsets &&
                                 starts_apart(d_offsets, B, kin, vin, kout, vout, n, kw, vw)
                             ? d_offsets : nullptr;
        const ShortCall c{kin, vin, kout, vout, n, kw, vw, offs, B, stream};
        auto go = [&](const auto& f) { return launch_short_block(c, (uint32_t)bits, f); };
        const hipError_t e = kw == 2 ? with_id64(d, B, 0u, ~0u, go) : go(id32(d, B, 0u, ~0u));
        if (e != hipSuccess || !d_offsets || offs) return hip_status(e);
        return wide_starts(kout, n, kw, B, d, d_offsets, stream);
    }
    uint32_t width[3], shift = 0;
    const int passes = large_passes((uint32_t)bits, vw != 0, true, n, width);
    const uint32_t* sk = kin;
    const uint32_t* sv = vin;
    for (int p = 0; p < passes; shift += width[p++]) {
        const uint32_t w = width[p];
        const bool to_out = ((passes - 1 - p) % 2) == 0;  // the last pass writes the output
        uint32_t* dk = to_out ? kout : ktmp;
        uint32_t* dv = vw ? (to_out ? vout : vtmp) : nullptr;
        const uint32_t mask = (1u << w) - 1u;
        gms_status st = wide_stages(s, sk, sv, dk, dv, n, kw, vw, 1u << w, d, B, shift, mask,
                                    nullptr, stream);
        if (st != GMS_SUCCESS) return st;
        sk = dk;
        sv = dv;
    }
    return d_offsets ? wide_starts(kout, n, kw, B, d, d_offsets, stream) : GMS_SUCCESS;
}

int wide_sort_passes(uint32_t key_words, uint32_t digit_bits, SortPass* p) {
    if (key_words == 1) return sort_schedule(digit_bits, p);
    if (digit_bits < 4 || digit_bits > 8) return 0;
    int k = 0;
    for (uint32_t s = 0; s < 64; s += digit_bits)
        p[k++] = {s, 64 - s < digit_bits ? 64 - s : digit_bits};
    return k;
}

gms_status run_wide_sort(Scratch& s, uint32_t* ktmp, uint32_t* vtmp, const uint32_t* kin,
                         const uint32_t* vin, uint32_t* kout, uint32_t* vout, uint32_t n,
                         uint32_t kw, uint32_t vw, uint32_t digit_bits, hipStream_t stream) {
    SortPass p[16];
    const int np = wide_sort_passes(kw, digit_bits, p);
    if (np == 0) return GMS_ERR_INVALID_ARG;
    if (short_one_block(n, 32u * kw, kw, vw)) {  // the whole key is the id
        const ShortCall c{kin, vin, kout, vout, n, kw, vw, nullptr, 0u, stream};
        return hip_status(kw == 2 ? launch_short_sort64(c)
                                  : launch_short_block(c, 32u, DigitOfF{AnyF{0u, ~0u, 0u, 0u, ~0u, ~0u}, 0u, ~0u}));
    }
    const uint32_t* sk = kin;
    const uint32_t* sv = vin;
    for (int i = 0; i < np; ++i) {
        // the last pass writes the output; the input is never written
        const bool to_out = ((np - 1 - i) % 2) == 0;
        uint32_t* dk = to_out ? kout : ktmp;
        uint32_t* dv = vw ? (to_out ? vout : vtmp) : nullptr;
        const gms_bucket_desc64 d{GMS_BUCKET_DIGIT, p[i].bits, p[i].shift};
        gms_status st = run_wide_multisplit(s, sk, sv, dk, dv, n, kw, vw, 1u << p[i].bits, d,
                                            nullptr, stream);
        if (st != GMS_SUCCESS) return st;
        sk = dk;
        sv = dv;
    }
    return GMS_SUCCESS;
}

}  // namespace gms
