// Multisplit into more than 256 buckets (up to kMaxBuckets).
//
// The reference's answer beyond 256 buckets is the reduced-bit sort (README,
// "Multisplit" item; src/kernels/RBsort/reduced_bit_sort.cuh:24-57 and its use
// in src/main/main_wms.cu:534-755): rank the elements by the bits of their
// bucket id with a stable radix sort, which equals the multisplit.  Here the
// id is never stored: LSD passes of this library's own multisplit rank by
// digits of f(key) (DigitOfF, computed from the key in every pass),
// carrying the keys and values themselves, ping-ponging through scratch so
// that the last pass writes the output and the input is never written.  The
// bucket starts, when asked, are read off the output: start[b] = first i with
// f(kout[i]) >= b.
#include "gms_internal.hpp"
#include "gms_kernels.hpp"

namespace gms {

gms_status large_scratch_alloc(LargeScratch& L, uint32_t n_capacity, uint32_t num_buckets,
                               bool temporaries) {
    large_scratch_free(L);
    const size_t words = std::max<size_t>(n_capacity, 1);
    if (temporaries) {
        if (hipMalloc((void**)&L.ktmp, words * sizeof(uint32_t)) != hipSuccess) L.ktmp = nullptr;
        if (hipMalloc((void**)&L.vtmp, words * sizeof(uint32_t)) != hipSuccess) L.vtmp = nullptr;
    }
    if (hipMalloc((void**)&L.offs, (size_t)num_buckets * sizeof(uint32_t)) != hipSuccess)
        L.offs = nullptr;
    if ((temporaries && (!L.ktmp || !L.vtmp)) || !L.offs) {
        large_scratch_free(L);
        return GMS_ERR_ALLOC;
    }
    L.cap = n_capacity;
    return GMS_SUCCESS;
}

void large_scratch_free(LargeScratch& L) {
    uint32_t** bufs[3] = {&L.ktmp, &L.vtmp, &L.offs};
    for (uint32_t** b : bufs) {
        if (*b) (void)hipFree(*b);
        *b = nullptr;
    }
    L.cap = 0;
}

// Passes of equal width where that pays, else 8 bits a pass.  On MI355X, whole
// call in us, 8 bits a pass against the rule, key-value / key-only:
//   13 bits  4M 64.4 / 59.5 -> 61.1 / 55.3 (7 + 6), 2^27 1101 / 749 -> 1063 / 743
//   17 bits  4M 86.6 / 78.9 -> 73.8 / 64.5 (9 + 8), 2^27 1629 / 1091 -> 1244 / 961
//   18 bits  4M 87.5 / 80.3 -> 79.4 / 77.4 (9 + 9), 2^27 1633 / 1095 -> 1352 / 1013
//   20 bits  4M 94.1 -> 89.7 (7 + 7 + 6), 2^27 1657 -> 1596; key-only 207 -> 213 at 20M,
//            so key-only keeps 8 + 8 + 4
//   11 bits  8 + 3: 4M 56.3 / 50.8, 20M 184 / 129 (6 + 5: 60.0 / 55.2, 183 / 140)
// 64-bit elements keep 8 bits a pass.
int large_passes(uint32_t bits, bool kv, bool wide, uint32_t (&width)[3]) {
    const uint32_t np = bits <= (wide ? 16u : 18u) ? 2u : 3u;
    const bool even = !wide && bits > 11u && (np == 2u || kv);
    for (uint32_t i = 0, left = bits; i < np; ++i) {
        width[i] = even ? (left + (np - i) - 1u) / (np - i) : (left < 8u ? left : 8u);
        left -= width[i];
    }
    return (int)np;
}

gms_status run_large_multisplit(LargeScratch& L, Scratch& s, const uint32_t* kin,
                                const uint32_t* vin, uint32_t* kout, uint32_t* vout, uint32_t n,
                                uint32_t B, gms_bucket_desc d, uint32_t* d_offsets,
                                hipStream_t stream) {
    if (n == 0) return d_offsets ? hip_status(launch_fill(d_offsets, 0u, B, stream)) : GMS_SUCCESS;
    if (n > L.cap || !L.ktmp || !L.vtmp) return GMS_ERR_CAPACITY;
    const AnyF base = AnyF::make(d.kind, d.param, d.width, B);
    const bool kv = vin != nullptr;
    const int bits = ceil_log2_u32(B);
    if (short_one_block(n, (uint32_t)bits, 1, kv)) {
        uint32_t* offs = B <= kShortBlockOffsets &&
                                 starts_apart(d_offsets, B, kin, vin, kout, vout, n, 1, kv)
                             ? d_offsets : nullptr;
        const ShortCall c{kin, vin, kout, vout, n, 1u, kv ? 1u : 0u, offs, B, stream};
        const hipError_t e = launch_short_block(c, (uint32_t)bits, DigitOfF{base, 0u, ~0u});
        if (e != hipSuccess || !d_offsets || offs) return hip_status(e);
        return hip_status(launch_bucket_starts<1>(kout, n, B, base, d_offsets, stream));
    }
    uint32_t width[3], shift = 0;
    const int passes = large_passes((uint32_t)bits, kv, false, width);
    const uint32_t* sk = kin;
    const uint32_t* sv = vin;
    for (int p = 0; p < passes; shift += width[p++]) {
        const uint32_t w = width[p];
        const bool to_out = ((passes - 1 - p) % 2) == 0;  // the last pass writes the output
        uint32_t* dk = to_out ? kout : L.ktmp;
        uint32_t* dv = kv ? (to_out ? vout : L.vtmp) : nullptr;
        const DigitOfF f{base, shift, (1u << w) - 1u};
        gms_status st = run_multisplit_digit(s, sk, sv, dk, dv, n, 1u << w, f, stream);
        if (st != GMS_SUCCESS) return st;
        sk = dk;
        sv = dv;
    }
    if (!d_offsets) return GMS_SUCCESS;
    return hip_status(launch_bucket_starts<1>(kout, n, B, base, d_offsets, stream));
}

}  // namespace gms
