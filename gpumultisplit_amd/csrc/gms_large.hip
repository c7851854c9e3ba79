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

// Passes of equal width where that measured faster, or on no key distribution more
// than a few percent slower than it is faster on others; else 8 bits a pass.  On
// MI355X, on buffers that change from call to call, time over that of 8 bits a
// pass, uniform / sorted / nine in ten keys equal:
//   12 bits  6 + 6: 2M .87 / .79 / .79, 2.2M 1.03 / 1.06 / 1.05, 2.6M .99 / 1.06 / 1.02; key-value 3M
//            .94 / 1.03 / 1.01, 4M .91 / 1.00 / .98, 9M .95 / 1.02 / 1.02, 2^25 .96 / .99 / 1.00;
//            key-only 3.5M 1.04 / 1.12 / 1.11, 9M .98 / 1.05 / 1.04
//   13 bits  7 + 6: 1.1M .96 / .96 / .96, 3M .91 / .97 / .97, 2^24 .98 / 1.00 / 1.00
//   14 bits  7 + 7: 2M 1.15 / 1.21 / 1.18, 3M .93 / .95 / .94, 9M key-only .97 / .98 / .98, key-value
//            .98 / 1.00 / .99; 2^27 key-only 1.08 / 1.07 / 1.04, key-value .95 / 1.10 / 1.04
//   17 bits  9 + 8: 1M .85 / .85 / .88, 9M .84 / .85 / .85, 2^27 key-value .77 / .81 / .81,
//            key-only .88 / 1.10 / 1.00 but 6 + 6 + 5 .95 / 1.00 / .97
//   18 bits  9 + 9: 1M .91 / .91 / .99, 9M .91 / .94 / .93, 2^27 key-value .83 / .90 / .91,
//            key-only .99 / 1.34 / 1.30 but 6 + 6 + 6 .95 / 1.03 / 1.00; 1.3M 1.05 / 1.06 / 1.23,
//            where 8-bit passes still take two launches and 9-bit ones do not
//   19 bits  7 + 6 + 6, key-value: 1.9M .93 / .93 / .94, 3M 1.03 / 1.02 / 1.05, 2^24 .96 / 1.01 / 1.02
//   20 bits  7 + 7 + 6, key-value: 1.3M .96 / .96 / .97, 1.9M 1.04 / 1.03 / 1.04, 9M 1.01 / 1.01 / 1.06
// 11 bits stay 8 + 3 (6 + 5: 9M 1.04 / 1.10 / 1.09), 64-bit elements at 8 bits a pass.
int large_passes(uint32_t bits, bool kv, bool wide, uint32_t n, uint32_t (&width)[3]) {
    uint32_t np = bits <= (wide ? 16u : 18u) ? 2u : 3u;
    bool even = false;
    if (!wide) {
        switch (bits) {
            case 12: even = n <= 1u << 21 || (kv && n >= 11u << 18); break;
            case 13: even = true; break;
            case 14: even = n > 1u << 21 && n < 1u << 26; break;
            case 17:
            case 18:
                even = !(bits == 18 && n > 1u << 20 && n <= 3u << 19);
                if (!even || (!kv && n >= kLongTileMin)) np = 3;
                break;
            case 19: even = kv && n <= 1u << 21; break;
            case 20: even = kv && n <= 3u << 19; break;
            default: break;
        }
    }
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
    const int passes = large_passes((uint32_t)bits, kv, false, n, width);
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

#ifdef GMS_HOST_EMULATION
// Test hook of the CPU emulation build only: the passes of a call.
extern "C" int gms_emu_large_passes(uint32_t bits, int kv, int wide, uint32_t n, uint32_t* width) {
    uint32_t w[3] = {0, 0, 0};
    const int np = gms::large_passes(bits, kv != 0, wide != 0, n, w);
    for (int i = 0; i < 3; ++i) width[i] = w[i];
    return np;
}
#endif
